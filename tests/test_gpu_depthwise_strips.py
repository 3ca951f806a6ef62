"""Every strip height of the matrix-core depthwise kernel (set_tile(-2, -rows)) against the vector-ALU kernels (set_tile(-3, 0)):
strips that the first input rows make, whole and broken steps, a last strip of any height, strips at both ends of the image."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,s", [(3, 1), (3, 2), (5, 1), (5, 2)])
@pytest.mark.parametrize("C,N,H,W", [(16, 2, 35, 21), (8, 3, 11, 70), (24, 5, 1, 4)])
@pytest.mark.parametrize("i8,act", [(True, 3), (True, 2), (False, 0)])
def test_strip_heights(hip, k, s, C, N, H, W, i8, act):
    rng = np.random.default_rng(k * 10 + s + C)
    conv = hip.conv(wq=rng.integers(-127, 128, (C, 1, k, k)).astype(np.int8), scale_in=host_scale_in(np.full(C, 30.0, np.float32), 20.0),
                    bias=rng.normal(0, 1, C).astype(np.float32), in_scale=20.0, out_scale=[9.0] if i8 else None, stride=(s, s),
                    pad=(k // 2, k // 2), groups=C, act=act, act_p0=0.1, out_kind=capi.OUT_I8 if i8 else capi.OUT_F32)
    x = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    conv.set_tile(-3, 0)
    want = conv.forward(x, capi.I8_P8, N, H, W)
    for rows in range(1, conv.out_hw(H, W)[0] + 1):
        conv.set_tile(-2, -rows)
        got = conv.forward(x, capi.I8_P8, N, H, W)
        assert hip.torch.equal(got.view(hip.torch.uint8), want.view(hip.torch.uint8)), rows
    conv.close()
