"""Pointwise layers on the launch that keeps its operands in registers (set_tile(-10, groups | pairs << 7)) against the implicit-GEMM
kernel (set_tile(-4, 0)), bit for bit: ends of reduction steps, of pixel groups and of channel pairs, every split and epilogue."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu

SHAPES = [  # C, K, N, H, W
    (8, 8, 1, 1, 1),
    (64, 40, 3, 5, 7),       # the last pair ends in its second octet; pixel groups across images
    (72, 96, 2, 9, 13),      # the second reduction step holds one octet
    (136, 264, 5, 4, 4),     # more pairs than a wave walks, images of one pixel group
    (256, 32, 9, 16, 17),
    (312, 72, 17, 3, 11),
    (384, 24, 2, 13, 13),
    (968, 136, 1, 5, 9),     # sixteen reduction steps, the last of one octet
]
# groups, pairs, and whether the waves of a workgroup share the reduction (needs two steps of 64 channels; otherwise at most four)
SPLITS = [(1, 1, 0), (2, 1, 0), (1, 3, 0), (2, 2, 0), (4, 1, 0), (4, 3, 0), (1, 1, 64), (1, 3, 64), (2, 1, 64), (2, 2, 64), (4, 3, 64), (0, 0, 0)]


def _can(C, groups, split):
    return groups == 0 or (C > 64 if split else C <= 256)


def _layer(hip, rng, C, K, act, i8):
    wq = rng.integers(-127, 128, (K, C, 1, 1)).astype(np.int8)
    return hip.conv(wq=wq, scale_in=host_scale_in(np.full(K, 60.0, np.float32) + rng.uniform(0, 1, K).astype(np.float32), 20.0),
                    bias=rng.normal(0, 1, K).astype(np.float32), in_scale=20.0, out_scale=[7.0] if i8 else None, act=act, act_p0=0.1,
                    out_kind=capi.OUT_I8 if i8 else capi.OUT_F32)


def _same(hip, got, want):
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert hip.torch.equal(a.view(hip.torch.uint8), b.view(hip.torch.uint8))


@pytest.mark.parametrize("C,K,N,H,W", SHAPES)
@pytest.mark.parametrize("i8", [True, False])
def test_splits_and_activations(hip, C, K, N, H, W, i8):
    rng = np.random.default_rng(C + K)
    x = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    for act in (0, 1, 2, 3):
        conv = _layer(hip, rng, C, K if i8 else K - 4, act, i8)  # (fp32: a last octet of which half exists)
        conv.set_tile(-4, 0)
        want = conv.forward(x, capi.I8_P8, N, H, W)
        for groups, pairs, split in SPLITS:
            if not _can(C, groups, split):
                continue
            conv.set_tile(-10, groups | split | pairs << 7)
            assert conv.launch_choice(capi.I8_P8, N, H, W, conv.default_out_layout())[0] == 10
            _same(hip, [conv.forward(x, capi.I8_P8, N, H, W)], [want])
        conv.close()


@pytest.mark.parametrize("C,K,N,H,W", SHAPES)
@pytest.mark.parametrize("act", [1, 2])
def test_sum_twin_and_joins(hip, C, K, N, H, W, act):
    rng = np.random.default_rng(C * 2 + K)
    x = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    other = hip.to_device(rng.normal(0, 3, N * K * H * W).astype(np.float32))
    conv = _layer(hip, rng, C, K, act, False)

    def everything():
        yield conv.forward_residual(x, capi.I8_P8, N, H, W, other, q_scale=9.0)
        yield conv.forward_residual(x, capi.I8_P8, N, H, W, other)
        yield conv.forward_twin(x, capi.I8_P8, N, H, W, 9.0, capi.ROUND_EXACT)
        for layout, odd, joined in ((capi.F32_P8, False, False), (capi.F32_P4, True, True)):
            for whole in (True, False):
                yield conv.forward_shuffle(x, N, H, W, other, layout, odd, joined, 9.0, capi.ROUND_SSE, whole=whole)
        if K > 8:
            yield conv.forward_residual_concat(x, N, H, W, other[:N * 8 * H * W], capi.F32_P8, 8, other[N * 8 * H * W:], capi.F32_P4, 9.0)

    conv.set_tile(-4, 0)
    want = list(everything())
    for groups, pairs, split in SPLITS:
        if not _can(C, groups, split) or (groups == 4 and not split):
            continue
        conv.set_tile(-10, groups | split | pairs << 7)
        for got, w in zip(everything(), want):
            _same(hip, got, w)
    conv.set_tile(-10, 4 | 1 << 7)  # four groups with a sum: refused, as more registers than there are
    with pytest.raises(capi.HipError):
        conv.forward_residual(x, capi.I8_P8, N, H, W, other)
    conv.close()


@pytest.mark.parametrize("C,K,N,H,W", [
    (256, 512, 2, 64, 63),    # below 4 << 20 results
    (256, 512, 2, 64, 64),    # that many
    (136, 1048, 1, 61, 67),   # few pixels, more channel pairs than a wave walks, the last of one octet
    (8, 8, 3, 421, 419),      # one channel pair, many pixels, the last group not full
    (48, 72, 7, 97, 89),
    (256, 4112, 1, 33, 31),
])
@pytest.mark.parametrize("act", [1, 3])
def test_split_of_many_clamped_results(hip, C, K, N, H, W, act):
    """The split that clamped int8 results have from 4 << 20 of them on."""
    rng = np.random.default_rng(C + K + W)
    x = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    conv = _layer(hip, rng, C, K, act, True)
    assert conv.launch_choice(capi.I8_P8, N, H, W, capi.I8_P8) == (10, 0)
    got = conv.forward(x, capi.I8_P8, N, H, W)
    conv.set_tile(-4, 0)
    _same(hip, [got], [conv.forward(x, capi.I8_P8, N, H, W)])
    conv.close()


@pytest.mark.parametrize("C", [24, 264])
def test_a_tile_of_no_launch_forces_nothing(hip, C):
    """set_tile(0, tn) leaves every choice automatic, whatever tn is: below 128 it names no channel pairs, 321 a split reduction."""
    rng = np.random.default_rng(C)
    K, N, H, W = 40, 2, 9, 11
    conv = _layer(hip, rng, C, K, 1, False)
    x = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    other = hip.to_device(rng.normal(0, 3, N * K * H * W).astype(np.float32))
    want = conv.forward(x, capi.I8_P8, N, H, W), conv.forward_shuffle(x, N, H, W, other, capi.F32_P8, False, True, 9.0)
    for tn in (1, 3, 1 | 64 | 2 << 7, 2 | 1 << 7):
        conv.set_tile(0, tn)
        assert conv.launch_choice(capi.I8_P8, N, H, W, conv.default_out_layout()) == (10, 0)
        _same(hip, [conv.forward(x, capi.I8_P8, N, H, W)], [want[0]])
        _same(hip, conv.forward_shuffle(x, N, H, W, other, capi.F32_P8, False, True, 9.0), want[1])
    conv.close()


def test_a_scale_per_output_channel_stays_with_the_other_kernels(hip):
    rng = np.random.default_rng(5)
    conv = hip.conv(wq=rng.integers(-127, 128, (16, 24, 1, 1)).astype(np.int8), scale_in=np.full(16, 1e-3, np.float32), in_scale=20.0,
                    out_scale=list(rng.uniform(5, 9, 16)), out_kind=capi.OUT_I8)
    assert conv.launch_choice(capi.I8_P8, 1, 7, 7, capi.I8_P8)[0] != 10
    conv.close()


@pytest.mark.parametrize("C", [72, 264])
@pytest.mark.parametrize("joined", [True, False])
def test_shuffle_of_a_result_beyond_32_bit_offsets(hip, C, joined):
    """2^28 values of the layer's own: the joined blob is 2 GiB, past the register kernel's offsets, each half by itself is not. What
    otter_hip_conv_join_launches promises holds for both."""
    torch = hip.torch
    K, N, H, W = 64, 2, 1449, 1449
    rng = np.random.default_rng(C)
    conv = _layer(hip, rng, C, K, 1, False)
    gen = torch.Generator(device=hip.device)
    gen.manual_seed(C)
    x = torch.randint(-127, 128, (N * C * H * W,), generator=gen, device=hip.device, dtype=torch.int8)
    other = torch.randn(N * K * H * W, generator=gen, device=hip.device)
    assert N * K * H * W * 8 >= 1 << 31 > N * K * H * W * 4
    assert conv.join_launches(capi.I8_P8, N, H, W) == 1
    got = conv.forward_shuffle(x, N, H, W, other, capi.F32_P8, False, joined, 9.0)
    conv.set_tile(-4, 0)
    want = conv.forward_shuffle(x, N, H, W, other, capi.F32_P8, False, joined, 9.0)
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))
    conv.close()


def test_more_channel_pairs_than_a_grid_dimension_holds(hip):
    rng = np.random.default_rng(9)
    C, K, N, H, W = 8, 32 * 65536 + 64, 1, 1, 3
    conv = _layer(hip, rng, C, K, 1, True)
    x = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    got = conv.forward(x, capi.I8_P8, N, H, W)
    conv.set_tile(-4, 0)
    _same(hip, [got], [conv.forward(x, capi.I8_P8, N, H, W)])
    conv.close()
