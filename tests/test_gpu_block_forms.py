"""otter_hip_conv_block_forward_form: a block in the form that the caller names. Every form that can run gives the three layers' result
bit for bit, from exactly the workspace that otter_hip_conv_block_form_workspace_bytes reports; the others are refused."""
import numpy as np
import pytest

from tensor_amd import capi
from test_gpu_block import make_block, one_by_one

pytestmark = pytest.mark.gpu

UNSUPPORTED, INVALID = -1, -2
BLOCKS = [  # cin, ce, cout, N, H, W, stride, f32_out, the forms that can run
    (64, 384, 64, 4, 14, 14, 1, True, (1, 2, 3)),     # otter_hip_conv_block_launches: 3
    (32, 192, 32, 64, 28, 28, 1, True, (1, 2, 3)),    # 1
    (24, 144, 24, 2, 56, 56, 1, False, (1, 2, 3)),
    (160, 960, 160, 64, 7, 7, 1, True, (1, 3)),       # too many channels for the shared launch; a workspace of partial sums
    (24, 144, 32, 2, 30, 44, 2, True, (2, 3)),        # stride 2: no single launch
    (16, 96, 24, 1, 9, 100, 1, False, (2, 3)),        # too wide for it
    (160, 192, 64, 2, 28, 28, 2, True, (3,)),
]


@pytest.fixture(autouse=True)
def automatic_choices(hip):
    before = hip.conv_block_set_always(0), hip.conv_block_set_pair(0)
    yield
    hip.conv_block_set_always(before[0])
    hip.conv_block_set_pair(before[1])


def refused(code, call):
    with pytest.raises(capi.HipError) as e:
        call()
    assert e.value.code == code


@pytest.mark.parametrize("cin,ce,cout,N,H,W,stride,f32_out,forms", BLOCKS)
def test_every_form_from_its_reported_workspace(hip, cin, ce, cout, N, H, W, stride, f32_out, forms):
    torch = hip.torch
    rng = np.random.default_rng(cin + ce + H)
    layers = make_block(hip, rng, cin, ce, cout, 3, f32_out, stride=stride)
    b = [l["conv"] for l in layers]
    x = hip.to_device(capi.pack_np(rng.integers(-127, 128, (N, cin, H, W)).astype(np.int8), 8))
    oh, ow = b[1].out_hw(H, W)
    res = hip.to_device(rng.normal(0, 1, N * cout * oh * ow).astype(np.float32)) if f32_out else None
    q_scale = 19.0 if f32_out else None
    want, want_q = one_by_one(hip, layers, x, N, H, W, res, q_scale)
    assert hip.conv_block_fastest(*b, N, H, W) in forms

    def reported(form):
        return hip.lib.otter_hip_conv_block_form_workspace_bytes(*[c.h for c in b], form, N, H, W)

    for form in (1, 2, 3):
        if form not in forms:
            assert reported(form) == 0, form
            refused(UNSUPPORTED, lambda: hip.conv_block_form(form, *b, x, N, H, W, residual=res, q_scale=q_scale))
            continue
        need = reported(form)
        room = torch.full((need + 4096,), 85, dtype=torch.int8, device=hip.device)
        for _ in range(2):
            got, got_q = hip.conv_block_form(form, *b, x, N, H, W, residual=res, q_scale=q_scale, workspace=room[:need])
            assert torch.equal(got, want.view(-1)), form
            assert not f32_out or torch.equal(got_q, want_q.view(-1)), form
            assert bool((room[need:] == 85).all()), form
        if need:
            refused(INVALID, lambda: hip.conv_block_form(form, *b, x, N, H, W, residual=res, q_scale=q_scale, workspace=room[:need - 1]))
    for form in (0, 4):
        assert reported(form) == 0, form
        refused(INVALID, lambda: hip.conv_block_form(form, *b, x, N, H, W, residual=res, q_scale=q_scale, workspace=room))
    for l in layers:
        l["conv"].close()


@pytest.mark.parametrize("f32_out,layout", [(True, capi.F32), (True, capi.F32_P8), (False, capi.I8)])
def test_other_layouts_are_not_for_the_single_launch(hip, f32_out, layout):
    rng = np.random.default_rng(layout)
    N, H, W = 3, 14, 14
    layers = make_block(hip, rng, 64, 384, 64, 3, f32_out)
    b = [l["conv"] for l in layers]
    x = hip.to_device(capi.pack_np(rng.integers(-127, 128, (N, 64, H, W)).astype(np.int8), 8))
    refused(UNSUPPORTED, lambda: hip.conv_block_form(1, *b, x, N, H, W, out_layout=layout))
    t = b[1].forward(b[0].forward(x, capi.I8_P8, N, H, W, capi.I8_P8), capi.I8_P8, N, H, W, capi.I8_P8)
    want = b[2].forward(t, capi.I8_P8, N, H, W, layout)
    for form in (2, 3):
        assert hip.torch.equal(hip.conv_block_form(form, *b, x, N, H, W, out_layout=layout)[0], want)
    for l in layers:
        l["conv"].close()
