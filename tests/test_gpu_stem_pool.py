"""otter_hip_conv_forward_maxpool: an image stem and the max pooling behind it in one launch. The results must be, bit for bit, those of the
layer, otter_hip_maxpool2d and the quantization one by one."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu


def stem(hip, rng, C, K, pad, act=2, p0=0.1, scale_in=None):
    w = rng.integers(-127, 128, (K, C, 3, 3)).astype(np.int8)
    si = host_scale_in(rng.uniform(200, 1500, K).astype(np.float32), 31.0) if scale_in is None else scale_in
    return hip.conv(wq=w, scale_in=si, bias=rng.normal(0, 0.4, K).astype(np.float32), in_scale=31.0, stride=(2, 2), pad=(pad, pad), act=act, act_p0=p0,
                    out_kind=capi.OUT_F32, in_round=capi.ROUND_EXACT)


def apart(hip, conv, x, layout, n, h, w, pad_value, q_scale, q_round):
    oh, ow = conv.out_hw(h, w)
    ph, pw = (oh - 1) // 2 + 1, (ow - 1) // 2 + 1
    y = conv.forward(x, layout, n, h, w, capi.F32_P4)
    p = hip.empty(n * conv.K * ph * pw, np.float32)
    hip._check(hip.lib.otter_hip_maxpool2d(hip.ptr(y), capi.F32_P4, n, conv.K, oh, ow, 3, 3, 2, 2, 1, 1, 1, 1, ph, pw, capi.C.c_float(pad_value), hip.ptr(p),
                                           capi.F32_P8, hip.stream()))
    q = hip.empty(n * conv.K * ph * pw, np.int8)
    scales = np.array([q_scale], np.float32)
    s = hip.to_device(scales)
    hip._check(hip.lib.otter_hip_quantize(hip.ptr(p), capi.F32_P8, n, conv.K, ph, pw, hip.ptr(s), 1, q_round, hip.ptr(q), capi.I8_P8, hip.stream()))
    hip.torch.cuda.synchronize()
    return p, q


@pytest.mark.parametrize("C,K,pad,act,n,h,w", [
    (3, 24, 1, 2, 2, 64, 64),      # whole strips, aligned rows
    (3, 24, 1, 2, 1, 37, 61),      # odd sides: the last window is over the border, rows of no whole units
    (3, 32, 0, 3, 2, 33, 130),     # no padding; more than one group of pooled columns and a clamp
    (1, 8, 1, 0, 3, 9, 7),         # fewer channels than a lane's four, half a tile
    (4, 64, 1, 1, 1, 20, 35),      # four tiles
    (2, 40, 0, 2, 2, 5, 4),        # a pooled row and column
    (3, 16, 1, 2, 1, 1, 1),        # one pixel: every window is border
    (3, 24, 1, 2, 1, 416, 416),
])
def test_one_launch_equals_the_layers(hip, C, K, pad, act, n, h, w):
    rng = np.random.default_rng(C + K + w)
    if h + 2 * pad < 3 or w + 2 * pad < 3:
        pytest.skip("no output")
    conv = stem(hip, rng, C, K, pad, act)
    for layout, x in ((capi.F32, rng.normal(0, 2, n * C * h * w).astype(np.float32)), (capi.I8, rng.integers(-127, 128, n * C * h * w).astype(np.int8))):
        xd = hip.to_device(x)
        for pad_value, q_round in ((0.0, capi.ROUND_SSE), (-np.inf, capi.ROUND_EXACT)):
            conv.set_tile(0, 0)
            p, q = apart(hip, conv, xd, layout, n, h, w, pad_value, 23.0, q_round)
            assert conv.maxpool_launches(layout, n, h, w) == 1
            for rows in (0, 1, 2, 4):  # pooled rows of a workgroup
                conv.set_tile(-13 if rows else 0, rows)
                got = conv.forward_maxpool(xd, layout, n, h, w, pad_value, 23.0, q_round)
                only = conv.forward_maxpool(xd, layout, n, h, w, pad_value, 23.0, q_round, whole=False)[1]
                alone = conv.forward_maxpool(xd, layout, n, h, w, pad_value)[0]
                hip.torch.cuda.synchronize()
                for k, (g, want) in enumerate(((got[0], p), (got[1], q), (only, q), (alone, p))):
                    assert hip.torch.equal(g, want), (layout, pad_value, rows, k)


def test_what_is_refused(hip):
    rng = np.random.default_rng(1)
    x = hip.empty(3 * 20 * 20, np.float32)
    si = np.full(24, 1e-3, np.float32)
    ok = stem(hip, rng, 3, 24, 1)
    assert ok.maxpool_launches(capi.F32, 1, 20, 20) == 1 and ok.maxpool_launches(capi.F32_P8, 1, 20, 20) == 2
    others = [stem(hip, rng, 3, 24, 1, scale_in=np.where(np.arange(24) == 5, v, si).astype(np.float32)) for v in (-1e-3, np.inf, np.nan)]  # not monotone
    others += [stem(hip, rng, 3, 24, 1, act=4), stem(hip, rng, 3, 20, 1), stem(hip, rng, 5, 24, 1)]
    for conv in others:
        assert conv.maxpool_launches(capi.F32, 1, 20, 20) == 2
        with pytest.raises(capi.HipError):
            conv.forward_maxpool(x, capi.F32, 1, 20, 20)
    for args, kw in (((capi.F32, 1, 20, 20), dict(pad_value=float("nan"))), ((capi.F32, 1, 20, 20), dict(q_scale=1.0, q_round_mode=9)),
                     ((capi.F32, 1, 20, 20), dict(whole=False))):
        with pytest.raises(capi.HipError):
            ok.forward_maxpool(x, *args, **kw)
