"""Max pooling and upsampling of blobs so large that a thread takes several channel packs, against the same images one at a time (one
pack per thread), bit for bit: pack counts that leave the last thread some of its packs only, unlike packs on the two sides, NaN and
infinities."""
import numpy as np
import pytest

from tensor_amd import capi

pytestmark = pytest.mark.gpu

MANY = 1 << 21  # values of a result from which on a thread takes several packs
LAYOUTS = [(capi.F32_P4, capi.F32_P4), (capi.F32_P8, capi.F32_P8), (capi.F32_P4, capi.F32_P8), (capi.F32_P8, capi.F32_P4)]


def _compare(hip, shape, out_hw, src, dst, run):
    n, c, h, w = shape
    rng = np.random.default_rng(c + h)
    x = rng.normal(0, 1, n * c * h * w).astype(np.float32)
    x[rng.integers(0, x.size, x.size // 50)] = rng.choice([np.nan, np.inf, -np.inf], x.size // 50)
    x = hip.to_device(x)
    assert n * c * out_hw[0] * out_hw[1] >= MANY > c * out_hw[0] * out_hw[1]
    got = run(x, shape).view(hip.torch.int32).reshape(-1)
    for i in range(n):
        part = c * h * w
        one = run(x[i * part:(i + 1) * part], (1, c, h, w)).view(hip.torch.int32).reshape(-1)
        assert hip.torch.equal(got[i * one.numel():(i + 1) * one.numel()], one), i


@pytest.mark.parametrize("src,dst", LAYOUTS)
@pytest.mark.parametrize("k,s,p,pad", [(3, 2, 1, 0.0), (3, 1, 1, -np.inf), (2, 2, 0, 0.0), (5, 1, 2, 0.0)])
def test_maxpool(hip, src, dst, k, s, p, pad):
    n, c, h, w = 8, 40, 41 * s, 199 * s
    oh, ow = (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
    _compare(hip, (n, c, h, w), (oh, ow), src, dst, lambda x, sh: hip.maxpool2d(x, src, sh, (k, k), (s, s), (p, p), (1, 1), (oh, ow), pad, dst))


@pytest.mark.parametrize("src,dst", LAYOUTS)
@pytest.mark.parametrize("mode,align,oh,ow", [(1, False, 78, 110), (2, False, 78, 110), (2, True, 77, 109), (2, False, 101, 83)])
def test_upsample(hip, src, dst, mode, align, oh, ow):
    _compare(hip, (8, 40, 39, 55), (oh, ow), src, dst, lambda x, sh: hip.upsample2d(x, src, sh, (oh, ow), mode, align, dst))
