"""Library.conv_block chooses among the forms of a block: whichever it takes, the three layers' result bit for bit, without a workspace, with
the one that otter_hip_conv_block_workspace_bytes reports, with less than that (refused as ever), and recorded into a graph."""
import numpy as np
import pytest

from tensor_amd import capi
from test_gpu_block import make_block, one_by_one
from test_gpu_block_forms import automatic_choices  # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu

BLOCKS = [  # cin, ce, cout, N, H, W, stride, f32_out, launches as ever, of the fastest form
    (128, 768, 128, 1, 13, 13, 1, True, 3, 2),    # fewer launches
    (64, 384, 64, 4, 8, 8, 1, True, 3, 2),
    (112, 672, 112, 33, 22, 22, 1, True, 1, 3),   # more, of blobs large enough
    (24, 144, 40, 49, 10, 9, 1, False, 1, 3),     # too small for more
    (24, 144, 24, 2, 14, 8, 2, False, 2, 2),
]


@pytest.mark.parametrize("cin,ce,cout,N,H,W,stride,f32_out,as_ever,fastest", BLOCKS)
def test_block_call(hip, cin, ce, cout, N, H, W, stride, f32_out, as_ever, fastest):
    torch = hip.torch
    rng = np.random.default_rng(cin + ce + H)
    layers = make_block(hip, rng, cin, ce, cout, 3, f32_out, stride=stride)
    b = [l["conv"] for l in layers]
    x = hip.to_device(capi.pack_np(rng.integers(-127, 128, (N, cin, H, W)).astype(np.int8), 8))
    oh, ow = b[1].out_hw(H, W)
    res = hip.to_device(rng.normal(0, 1, N * cout * oh * ow).astype(np.float32)) if f32_out else None
    q_scale = 19.0 if f32_out else None
    want, want_q = one_by_one(hip, layers, x, N, H, W, res, q_scale)

    def same(got, got_q):
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
        assert q_scale is None or torch.equal(got_q, want_q)

    reported = hip.lib.otter_hip_conv_block_workspace_bytes(*[c.h for c in b], N, H, W)
    for room in (None, torch.empty(max(reported, 1), dtype=torch.int8, device=hip.device), torch.empty(64 << 20, dtype=torch.int8, device=hip.device)):
        same(*hip.conv_block(*b, x, N, H, W, residual=res, q_scale=q_scale, workspace=room))
    if as_ever > 1:
        with pytest.raises(capi.HipError):
            hip.conv_block(*b, x, N, H, W, residual=res, q_scale=q_scale, workspace=torch.empty(64, dtype=torch.int8, device=hip.device))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = hip.conv_block(*b, x, N, H, W, residual=res, q_scale=q_scale)
    for _ in range(3):
        out[0].zero_()
        g.replay()
        torch.cuda.synchronize()
        same(*out)
    assert (hip.conv_block_launches(*b, N, H, W), hip.conv_block_fastest(*b, N, H, W)) == (as_ever, fastest)
