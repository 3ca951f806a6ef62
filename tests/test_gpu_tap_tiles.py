"""Every tile of the launch that deals the reduction to the waves of a workgroup (set_tile(-8, tile)) against the implicit-GEMM kernel
(set_tile(-4, 0)), bit for bit: every number of steps that a wave can be left with behind its last whole trip, and windows that leave the
image on each side, by more than their own size, with 31 taps in a row and in a column."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu

TILES = range(7)
STEPS = [(8, (1, 1)), (64, (1, 2)), (64, (1, 3)), (40, (3, 3)), (64, (2, 4)), (64, (3, 3)), (64, (3, 4)), (104, (3, 3)), (136, (3, 3)), (88, (5, 5)),
         (264, (3, 3)), (328, (3, 3))]  # 1 to 47 steps
WINDOWS = [  # kernel, stride, pad, dilation, image
    ((1, 31), (1, 1), (0, 15), (1, 1), (3, 5)),
    ((31, 1), (1, 1), (15, 0), (1, 1), (6, 2)),
    ((5, 6), (1, 2), (9, 4), (1, 1), (3, 7)),    # rows of windows entirely above and below the image
    ((6, 5), (2, 1), (4, 9), (1, 1), (7, 2)),    # columns of windows entirely beside it
    ((3, 3), (3, 3), (1, 1), (1, 1), (1, 1)),
    ((4, 7), (1, 1), (3, 6), (2, 1), (6, 9)),    # dilated in one direction only
    ((2, 3), (1, 1), (0, 1), (1, 3), (8, 11)),
]


def _check(hip, C, kernel, image, stride=(1, 1), pad=(0, 0), dil=(1, 1), K=72, N=3):
    rng = np.random.default_rng(C + kernel[0] * 100 + kernel[1])
    H, W = image
    q = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    f = hip.to_device(rng.uniform(-8, 8, N * C * H * W).astype(np.float32))
    wq = rng.integers(-127, 128, (K, C) + kernel).astype(np.int8)
    scale = host_scale_in(np.full(K, 60.0, np.float32) + rng.uniform(0, 1, K).astype(np.float32), 20.0)
    bias = rng.normal(0, 1, K).astype(np.float32)
    for i8, act in ((True, 1), (False, 2)):
        conv = hip.conv(wq=wq, scale_in=scale, bias=bias, in_scale=20.0, out_scale=[0.7] if i8 else None, stride=stride, pad=pad, dil=dil, act=act,
                        act_p0=0.1, out_kind=capi.OUT_I8 if i8 else capi.OUT_F32)
        for x, layout in ((q, capi.I8_P8), (f, capi.F32_P8)):
            conv.set_tile(-4, 0)
            want = conv.forward(x, layout, N, H, W)
            for tile in TILES:
                if layout == capi.F32_P8 and tile == 4:  # (int8 only)
                    continue
                conv.set_tile(-8, tile)
                assert conv.launch_choice(layout, N, H, W, conv.default_out_layout()) == (8, tile)
                got = conv.forward(x, layout, N, H, W)
                assert hip.torch.equal(got.view(hip.torch.uint8), want.view(hip.torch.uint8)), (tile, layout, i8)
        conv.close()


@pytest.mark.parametrize("C,kernel", STEPS)
def test_every_remainder_of_steps(hip, C, kernel):
    _check(hip, C, kernel, (7, 9), pad=(kernel[0] // 2, kernel[1] // 2))


@pytest.mark.parametrize("kernel,stride,pad,dil,image", WINDOWS)
def test_windows_at_the_edges(hip, kernel, stride, pad, dil, image):
    _check(hip, 16, kernel, image, stride=stride, pad=pad, dil=dil)
