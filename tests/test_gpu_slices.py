"""otter_hip_conv_forward_slice, otter_hip_upsample2d_slice: a layer's result quantized into its channels of a Byte8 blob. Bit for bit the
layer's fp32 result and otter_hip_quantize of it, and nothing written beside those channels."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu
BEFORE, BEHIND, FILL = 16, 8, 99  # channels beside the slice, and what they hold


def quantized(hip, y, layout, n, c, h, w, scale, mode):
    q, s = hip.empty(n * c * h * w, np.int8), hip.to_device(np.array([scale], np.float32))
    hip._check(hip.lib.otter_hip_quantize(hip.ptr(y), layout, n, c, h, w, hip.ptr(s), 1, mode, hip.ptr(q), capi.I8_P8, hip.stream()))
    hip.torch.cuda.synchronize()
    return q.cpu().numpy()


def check_slice(hip, blob, want, n, c, h, w):
    hip.torch.cuda.synchronize()
    got = blob.cpu().numpy().reshape(n, (BEFORE + c + BEHIND) // 8, h * w * 8)
    np.testing.assert_array_equal(got[:, BEFORE // 8:(BEFORE + c) // 8].reshape(-1), want)
    assert (got[:, :BEFORE // 8] == FILL).all() and (got[:, (BEFORE + c) // 8:] == FILL).all()


def check_conv(hip, conv, rng, n, h, w, twin):
    C, K, total = conv.C, conv.K, BEFORE + conv.K + BEHIND
    oh, ow = conv.out_hw(h, w)
    x = hip.to_device(rng.integers(-127, 128, n * C * h * w).astype(np.int8))
    y = conv.forward(x, capi.I8_P8, n, h, w, capi.F32_P4)
    assert conv.slice_launches(capi.I8_P8, n, h, w, total, twin) == 1
    for scale, mode, other in ((17.0, capi.ROUND_SSE, capi.ROUND_EXACT), (400.0, capi.ROUND_EXACT, capi.ROUND_SSE)):
        blob = hip.to_device(np.full(n * total * oh * ow, FILL, np.int8))
        t = conv.forward_slice(x, capi.I8_P8, n, h, w, blob, total, BEFORE, scale, mode, 29.0 if twin else None, other)
        check_slice(hip, blob, quantized(hip, y, capi.F32_P4, n, K, oh, ow, scale, mode), n, K, oh, ow)
        if twin:
            np.testing.assert_array_equal(t.cpu().numpy(), quantized(hip, y, capi.F32_P4, n, K, oh, ow, 29.0, other))


@pytest.mark.parametrize("C,K,act,p0,n,h,w", [
    (8, 8, 0, 0.0, 1, 1, 1), (64, 40, 1, 0.0, 2, 7, 9), (128, 128, 2, 0.1, 3, 13, 13), (96, 72, 3, 0.0, 1, 26, 26), (256, 136, 2, 0.1, 1, 5, 3),
    (512, 64, 2, 0.1, 2, 13, 11), (1024, 256, 0, 0.0, 1, 13, 13), (64, 64, 2, 0.1, 16, 52, 52), (40, 24, 2, 1.5, 2, 30, 33),
])
def test_pointwise(hip, C, K, act, p0, n, h, w):
    rng = np.random.default_rng(C + K + w)
    conv = hip.conv(wq=rng.integers(-127, 128, (K, C, 1, 1)).astype(np.int8), bias=rng.normal(0, 0.4, K).astype(np.float32), in_scale=31.0,
                    scale_in=host_scale_in(rng.uniform(200, 1500, K).astype(np.float32), 31.0), act=act, act_p0=p0, out_kind=capi.OUT_F32)
    if p0 > 1:  # (a slope that the packed results' clamp does not hold for: the layer is left to its own launch, as before)
        assert conv.slice_launches(capi.I8_P8, n, h, w, BEFORE + K + BEHIND) == 2
        return
    for twin in (False, True):
        check_conv(hip, conv, rng, n, h, w, twin)


@pytest.mark.parametrize("C,ks,act,p0,n,h,w", [
    (8, 3, 0, 0.0, 1, 3, 3), (40, 3, 1, 0.0, 2, 7, 9), (128, 3, 2, 0.1, 3, 13, 13), (64, 5, 3, 0.0, 2, 26, 26), (24, 5, 2, 0.1, 5, 5, 4),
    (64, 3, 2, 0.1, 16, 52, 52), (16, 3, 3, 0.0, 1, 30, 131),
])
def test_depthwise(hip, C, ks, act, p0, n, h, w):
    rng = np.random.default_rng(C + ks + w)
    conv = hip.conv(wq=rng.integers(-127, 128, (C, 1, ks, ks)).astype(np.int8), groups=C, pad=(ks // 2, ks // 2), in_scale=31.0, act=act, act_p0=p0,
                    bias=rng.normal(0, 0.4, C).astype(np.float32), scale_in=host_scale_in(rng.uniform(40, 300, C).astype(np.float32), 31.0), out_kind=capi.OUT_F32)
    check_conv(hip, conv, rng, n, h, w, False)
    assert conv.slice_launches(capi.I8_P8, n, h, w, BEFORE + C + BEHIND, True) == 2


@pytest.mark.parametrize("c,n,h,w,oh,ow", [(8, 1, 2, 2, 4, 4), (24, 2, 7, 5, 14, 10), (128, 4, 26, 26, 52, 52), (32, 1, 9, 13, 20, 7)])
@pytest.mark.parametrize("layout", [capi.F32_P4, capi.F32_P8])
def test_upsample(hip, c, n, h, w, oh, ow, layout):
    x = hip.to_device(np.random.default_rng(c + w).normal(0, 3, n * c * h * w).astype(np.float32))
    total = BEFORE + c + BEHIND
    for mode in (1, 2):
        y = hip.upsample2d(x, layout, (n, c, h, w), (oh, ow), mode, False, capi.F32_P8)
        for scale, rounding in ((17.0, capi.ROUND_SSE), (60.0, capi.ROUND_EXACT)):
            blob = hip.to_device(np.full(n * total * oh * ow, FILL, np.int8))
            hip.upsample2d_slice(x, layout, (n, c, h, w), (oh, ow), mode, False, blob, total, BEFORE, scale, rounding)
            check_slice(hip, blob, quantized(hip, y, capi.F32_P8, n, c, oh, ow, scale, rounding), n, c, oh, ow)


def test_an_empty_batch(hip):
    conv = hip.conv(wq=np.ones((16, 16, 1, 1), np.int8), scale_in=np.full(16, 0.01, np.float32), in_scale=31.0, out_kind=capi.OUT_F32)
    x, blob = hip.to_device(np.zeros(16, np.int8)), hip.to_device(np.full(32, FILL, np.int8))
    conv.forward_slice(x, capi.I8_P8, 0, 5, 5, blob, 32, 16, 10.0)
    hip.upsample2d_slice(x, capi.F32_P8, (0, 16, 5, 5), (10, 10), 1, False, blob, 32, 16, 10.0, capi.ROUND_SSE)
    assert (blob == FILL).all()
    with pytest.raises(capi.HipError):
        conv.forward_slice(x, capi.I8_P8, 0, 5, 5, blob, 32, 24, 10.0)


def test_what_is_refused(hip):
    rng = np.random.default_rng(5)
    conv = hip.conv(wq=rng.integers(-127, 128, (16, 16, 1, 1)).astype(np.int8), scale_in=np.full(16, 0.01, np.float32), in_scale=31.0, out_kind=capi.OUT_F32)
    x, blob = hip.to_device(np.zeros(16 * 25, np.int8)), hip.to_device(np.zeros(32 * 25, np.int8))
    for total, first in ((32, 4), (32, 24), (32, -8), (20, 0)):
        with pytest.raises(Exception):
            conv.forward_slice(x, capi.I8_P8, 1, 5, 5, blob, total, first, 10.0)
    assert conv.slice_launches(capi.F32_P8, 1, 5, 5, 32) == 2
    xf = hip.to_device(np.zeros(16 * 25, np.float32))
    with pytest.raises(Exception):
        hip.upsample2d_slice(xf, capi.F32, (1, 16, 5, 5), (10, 10), 1, False, blob, 32, 0, 10.0, capi.ROUND_SSE)  # (not packed)
    with pytest.raises(Exception):
        hip.upsample2d_slice(xf, capi.F32_P8, (1, 16, 5, 5), (1, 1), 1, False, blob, 32, 24, 10.0, capi.ROUND_SSE)
