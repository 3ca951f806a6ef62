"""The launch that the cost models choose for a layer, at shapes where each form was measured well ahead of the others (us: the
family's own launch / the one that deals the reduction to its waves / the one on staged rows, best tile of each) and where an
earlier fit chose a slow one."""
import numpy as np
import pytest

from tensor_amd import capi

pytestmark = pytest.mark.gpu

FAMILY, TAP, ROWS = 0, 8, 9
CASES = [
    # cin, cout, kernel, stride, groups, n, h, w, fp32 blob, fp32 result, launches that are right
    (232, 344, 3, 2, 1, 30, 57, 66, False, False, (FAMILY, TAP)),    # 64 / 62, its widest tile 112 / 64
    (232, 112, 3, 2, 1, 16, 124, 187, False, False, (FAMILY, TAP)),  # 61 / 67, its widest tile 106 / 68
    (200, 280, 3, 2, 1, 7, 141, 141, False, False, (FAMILY, TAP)),   # 54 / 52, its widest tile 86 / 62
    (128, 1280, 1, 1, 1, 1, 29, 29, True, True, (TAP,)),             # 15.7 / 5.5
    (88, 624, 1, 1, 1, 12, 10, 14, True, True, (TAP,)),              # 9.5 / 5.4
    (216, 136, 1, 1, 1, 11, 38, 38, True, True, (FAMILY,)),          # 6.8 / 10.5
    (256, 256, 3, 1, 8, 64, 28, 28, False, False, (ROWS,)),          # 22.6 / 30 / 13.9
    (336, 184, 3, 1, 1, 1, 13, 13, False, False, (TAP,)),            # 22.7 / 4.5
    (24, 32, 3, 1, 1, 42, 205, 224, True, False, (ROWS,)),           # 107 / 180 / 71
    (56, 40, 3, 1, 1, 7, 123, 123, False, False, (FAMILY,)),         # 8.0 / 11.9 / 8.6
    (64, 64, 3, 1, 1, 8, 224, 224, False, False, (FAMILY,)),         # 22.4 / 38.7 / 23.4, with the tile that its model names 25.3
    (504, 144, 3, 1, 1, 2, 141, 141, False, False, (ROWS,)),         # 72 / 73 / 45
    (88, 32, 3, 1, 1, 38, 81, 65, False, False, (ROWS,)),            # 17.0 / 24.9 / 12.1
    (232, 224, 3, 1, 1, 2, 132, 132, False, True, (ROWS,)),          # 41 / 43 / 28
]


@pytest.mark.parametrize("cin,cout,k,stride,groups,n,h,w,f32in,f32out,right", CASES)
def test_launch_choice(hip, cin, cout, k, stride, groups, n, h, w, f32in, f32out, right):
    rng = np.random.default_rng(0)
    conv = hip.conv(wq=rng.integers(-127, 128, (cout, cin // groups, k, k)).astype(np.int8),
                    scale_in=np.full(cout, 1e-3, np.float32), bias=np.zeros(cout, np.float32), in_scale=40.0,
                    out_scale=None if f32out else [20.0], stride=(stride, stride), pad=(k // 2, k // 2), groups=groups, act=1,
                    out_kind=capi.OUT_F32 if f32out else capi.OUT_I8)
    choice = conv.launch_choice(capi.F32_P8 if f32in else capi.I8_P8, n, h, w, capi.F32_P4 if f32out else capi.I8_P8)
    assert choice[0] in right, choice
    if choice[0] == TAP and stride == 2:
        assert choice[1] != 4, "the widest tile reads such a blob from beyond the L2 for every tap"
    conv.close()
