"""CPU: the plan of the launch that stages input rows in LDS (host arithmetic of the GPU library, no GPU needed). The LDS it asks
for must be what its rows and columns add up to, in whole numbers that do not wrap, and the rows at least as many as any tile
touches."""
import ctypes as C

import pytest

from tensor_amd import capi

LDS = 64 * 1024


def rows_plan(cin, cout, groups, kernel, stride, pad, dil, n, h, w, pixels):
    d = capi.ConvDesc(cin, cout, kernel[0], kernel[1], stride, stride, pad[0], pad[1], dil[0], dil[1], groups, 0, 0.0, capi.OUT_I8, 0, 0)
    plan = (C.c_int * 6)()
    rc = capi.load_cdll().otter_hip_conv_rows_plan(C.byref(d), n, h, w, pixels, plan)
    return dict(zip(("strips", "strip_w", "rows", "pairs", "plane", "lds"), plan)) if rc == 0 else None


def check(p, cin, groups, kernel, stride, pad, dil, h, w, pixels):
    oh, ow = (h + 2 * pad[0] - dil[0] * (kernel[0] - 1) - 1) // stride + 1, (w + 2 * pad[1] - dil[1] * (kernel[1] - 1) - 1) // stride + 1
    assert p["strips"] * p["strip_w"] >= ow > (p["strips"] - 1) * p["strip_w"]
    # a row holds a strip's input columns and one in front, in pairs
    assert 2 * p["pairs"] >= (p["strip_w"] - 1) * stride + (kernel[1] - 1) * dil[1] + 1 + 1
    # the rows of a tile, wherever it starts: from the first output row's window to the last one's, in padded images laid out one
    # after the other
    vh, sw = (oh - 1) * stride + (kernel[0] - 1) * dil[0] + 1, p["strip_w"]
    need = 0
    for t0 in {t % (oh * sw) for t in range(0, 40 * pixels, pixels)} if oh * sw < 4000 else {0, pixels}:
        def row(t):
            return t // (oh * sw) * vh + t % (oh * sw) // sw * stride
        need = max(need, row(t0 + pixels - 1) + (kernel[0] - 1) * dil[0] + 1 - row(t0))
    assert p["rows"] >= need
    octets = -(-(cin // groups // 8) // -(-(cin // groups // 8) // 8))
    assert p["plane"] >= p["rows"] * p["pairs"] * 16 and p["plane"] % 128 == 64
    table = (kernel[0] * kernel[1] * 8 + 7) // 8 * 32 + (p["rows"] + 1) // 2 * 16
    assert p["lds"] == table + octets * p["plane"] <= LDS


@pytest.mark.parametrize("pixels", [128, 256])
@pytest.mark.parametrize("cin,groups,k,stride,dil,h,w", [(256, 8, 3, 1, 1, 28, 28), (8, 1, 5, 1, 1, 113, 113), (16, 1, 3, 1, 2, 204, 204),
                                                         (88, 1, 3, 2, 1, 57, 43), (24, 1, 5, 1, 1, 7, 7), (64, 1, 3, 1, 1, 1, 1),
                                                         (16, 1, 3, 3, 1, 20, 31), (16, 1, 3, 1, 40, 30, 30)])
def test_plan_holds_every_tile(cin, groups, k, stride, dil, h, w, pixels):
    pad = dil * (k // 2)
    p = rows_plan(cin, cin, groups, (k, k), stride, (pad, pad), (dil, dil), 3, h, w, pixels)
    if p is None:
        assert dil == 40 or stride == 3 or h == 1  # (too much LDS)
        return
    check(p, cin, groups, (k, k), stride, (pad, pad), (dil, dil), h, w, pixels)


def test_dilations_in_the_thousands():
    """Rows times columns times 16 bytes pass 2^31 there, and 2^32 exactly for some: no such plan may be taken for a small one."""
    refused = 0
    for pixels in (128, 256):
        for dh in list(range(4080, 4100)) + list(range(8170, 8196)) + [16384, 30000]:
            for dw in (dh, 8160, 16300, 16340, 16350, 16352, 16358, 16360, 16368, 16374, 16376, 16380, 32760):
                p = rows_plan(8, 8, 1, (3, 3), 1, (dh, dw), (dh, dw), 1, 64, 32, pixels)
                if p is None:
                    refused += 1
                else:
                    check(p, 8, 1, (3, 3), 1, (dh, dw), (dh, dw), 64, 32, pixels)
    assert refused > 0
