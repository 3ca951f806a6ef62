"""Depthwise layers on an fp32 Float8 blob as one launch where that is the faster form: 5x5 windows, and 3x3 on images of fewer than 17 columns. The bits are
those of a quantize pass and the int8 kernel (set_tile(-6, 0))."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu

SHAPES = [
    # C, k, stride, pad, N, H, W
    (16, 3, 1, 1, 2, 7, 7), (8, 3, 2, 1, 3, 9, 16), (24, 3, 1, 0, 1, 3, 3), (8, 3, 1, 1, 40, 40, 15),  # the last: strips of several rows, walked up and down
    (8, 5, 1, 2, 2, 5, 1), (16, 5, 1, 2, 1, 13, 13), (8, 5, 2, 2, 2, 12, 17), (8, 5, 1, 2, 1, 70, 32), (24, 5, 1, 2, 1, 31, 33), (8, 5, 1, 2, 1, 9, 64),
    (8, 5, 2, 2, 1, 33, 65), (8, 5, 1, 2, 1, 20, 97), (16, 5, 2, 1, 1, 41, 128), (64, 5, 1, 2, 10, 24, 20), (64, 5, 2, 2, 10, 48, 20), (8, 5, 2, 1, 1, 3, 3),
]


@pytest.mark.parametrize("C,k,stride,pad,N,H,W", SHAPES)
def test_one_launch_equals_two(hip, C, k, stride, pad, N, H, W):
    rng = np.random.default_rng(C + 10 * k + W)
    in_scale = np.float32(40.0)
    x = (rng.integers(-330, 331, (N, C, H, W)) / np.float32(2) / in_scale).astype(np.float32)  # half of them ties, some saturated
    flat = x.reshape(-1)
    flat[::11] = rng.normal(0, 1, flat[::11].size)
    flat[3::13] = np.nextafter(np.float32(0.5), np.float32(0)) / in_scale
    w = rng.integers(-127, 128, (C, 1, k, k)).astype(np.int8)
    ws = rng.uniform(40, 400, C).astype(np.float32)
    blob = hip.to_device(capi.pack_np(x, 8))
    for act, out_scale, layout in ((3, 127 / 6, capi.I8_P8), (3, 9.0, capi.I8_P8), (1, 0.7, capi.I8_P8), (0, 1.1, capi.I8_P8), (2, 1.3, capi.I8_P8),
                                   (2, None, capi.F32_P8), (3, None, capi.F32_P4)):
        conv = hip.conv(wq=w, scale_in=host_scale_in(ws, in_scale), bias=rng.normal(0, 0.4, C).astype(np.float32), in_scale=float(in_scale), groups=C, act=act, act_p0=0.1,
                        stride=(stride, stride), pad=(pad, pad), out_kind=capi.OUT_F32 if out_scale is None else capi.OUT_I8,
                        out_scale=None if out_scale is None else [out_scale], in_round=capi.ROUND_EXACT if act == 2 else capi.ROUND_SSE)
        oh, ow = conv.out_hw(H, W)
        one = hip.empty(N * C * oh * ow, np.float32 if out_scale is None else np.int8).fill_(77)
        # (a call without a workspace: it is refused where a quantize pass would need one)
        assert hip.lib.otter_hip_conv_forward(conv.h, hip.ptr(blob), capi.F32_P8, N, H, W, hip.ptr(one), layout, None, 0, hip.stream()) == 0
        conv.set_tile(-6, 0)
        two = conv.forward(blob, capi.F32_P8, N, H, W, layout)
        assert hip.torch.equal(one.view(hip.torch.uint8), two.view(hip.torch.uint8)), (act, out_scale, layout)
        conv.close()


def test_two_launches_stay_where_they_are_faster(hip):
    """Many planes of narrow images, of which a wave's lanes hold little: a call without a workspace is refused there, as it was."""
    C, n, side = 840, 56, 9
    rng = np.random.default_rng(1)
    conv = hip.conv(wq=rng.integers(-127, 128, (C, 1, 5, 5)).astype(np.int8), scale_in=np.full(C, 1e-3, np.float32), bias=None, in_scale=30.0, groups=C, act=0,
                    pad=(2, 2), out_kind=capi.OUT_I8, out_scale=[20.0])
    x = hip.to_device(rng.normal(0, 1, n * C * side * side).astype(np.float32))
    out = hip.empty(n * C * side * side, np.int8)
    assert hip.lib.otter_hip_conv_forward(conv.h, hip.ptr(x), capi.F32_P8, n, side, side, hip.ptr(out), capi.I8_P8, None, 0, hip.stream()) < 0
    conv.forward(x, capi.F32_P8, n, side, side)
    conv.close()
