"""Every tile of the k x k launch on staged rows (set_tile(-9, tile)) against the implicit-GEMM kernel (set_tile(-4, 0)), bit for bit: rows
shorter and longer than the 16 pixels from which a lane walks on instead of dividing, images that a tile runs over, column strips, output
channels beyond the threads of a workgroup and those whose constants it holds, and reductions of more than one stage whose weights are asked for ahead."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu

TILES = range(4)
LAYERS = [  # N, C, H, W, K, k, stride, pad, dilation, groups
    (3, 8, 9, 15, 16, 3, 1, 1, 1, 1),      # output rows of 15, 16 and 17 pixels
    (3, 8, 9, 16, 24, 3, 1, 1, 1, 1),
    (9, 24, 1, 17, 40, 3, 1, 1, 1, 1),     # an image a row: one more ends with every row
    (40, 16, 2, 16, 8, 3, 1, 1, 1, 1),
    (2, 40, 33, 33, 36, 3, 2, 1, 1, 1),    # (K % 8 == 4)
    (2, 16, 12, 50, 72, 5, 1, 3, 2, 1),    # odd pad, dilated
    (1, 8, 7, 200, 16, 3, 1, 1, 1, 1),     # strips
    (64, 8, 33, 33, 520, 3, 1, 1, 1, 1),   # a workgroup walks as many row blocks as it holds the constants of
    (2, 64, 20, 20, 96, 5, 1, 2, 1, 1),    # 25 steps of one stage
    (3, 200, 17, 19, 72, 3, 1, 1, 1, 1),   # four stages, 29 steps
    (70, 256, 5, 5, 40, 3, 1, 1, 1, 1),
    (2, 96, 19, 23, 144, 3, 1, 1, 1, 2),   # groups
    (2, 64, 18, 18, 64, 3, 1, 1, 1, 8),
    (1, 40, 30, 60, 64, 5, 2, 2, 1, 1),    # rows up to the last of a workgroup's 64 KB of LDS, and the constants beyond them
]


@pytest.mark.parametrize("layer", LAYERS)
def test_every_tile(hip, layer):
    N, C, H, W, K, k, stride, pad, dil, groups = layer
    rng = np.random.default_rng(C + 100 * W + K)
    q = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    f = hip.to_device(rng.uniform(-8, 8, N * C * H * W).astype(np.float32))
    wq = rng.integers(-127, 128, (K, C // groups, k, k)).astype(np.int8)
    scale = host_scale_in(np.full(K, 60.0, np.float32) + rng.uniform(0, 1, K).astype(np.float32), 20.0)
    bias = rng.normal(0, 1, K).astype(np.float32)
    for i8, act in ((True, 1), (True, 2), (True, 0), (False, 1)):
        if i8 and K % 8:
            continue
        # (output scales that differ from channel to channel)
        conv = hip.conv(wq=wq, scale_in=scale, bias=bias, in_scale=20.0, out_scale=list(np.linspace(0.4, 2, K)) if i8 else None, stride=(stride, stride),
                        pad=(pad, pad), dil=(dil, dil), groups=groups, act=act, act_p0=0.1, out_kind=capi.OUT_I8 if i8 else capi.OUT_F32)
        for x, layout in ((q, capi.I8_P8), (f, capi.F32_P8)):
            conv.set_tile(-4, 0)
            want = conv.forward(x, layout, N, H, W)
            for tile in TILES:
                conv.set_tile(-9, tile)
                assert conv.launch_choice(layout, N, H, W, conv.default_out_layout()) == (9, tile)
                got = conv.forward(x, layout, N, H, W)
                assert hip.torch.equal(got.view(hip.torch.uint8), want.view(hip.torch.uint8)), (tile, layout, i8, act)
        conv.close()
