"""otter_hip_conv_pair_forward: two pointwise layers in one launch. The results must be, bit for bit, what the two layers give one by
one, with a shuffle between them as with otter_hip_conv_forward_shuffle."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu

CASES = [
    # C, K, K2, N, H, W, first act, second act
    (88, 88, 88, 2, 52, 52, 2, 2),       # two reduction steps, three pairs for four waves
    (176, 176, 176, 3, 26, 26, 2, 2),    # three steps, six pairs
    (352, 352, 352, 2, 13, 13, 2, 0),    # six steps: two rounds of weights
    (576, 96, 576, 3, 14, 14, 0, 3),     # nine steps, then two
    (960, 160, 960, 2, 7, 7, 0, 3),      # the longest reduction; 49 pixels an image
    (128, 128, 112, 3, 7, 7, 2, 0),
    (8, 8, 8, 1, 1, 1, 1, 1),            # one pixel, a quarter of a pair
    (24, 40, 16, 5, 3, 5, 0, 2),         # a lane's channels past the last ones
    (64, 264, 72, 1, 9, 11, 3, 1),       # nine pairs
]


def layer(hip, rng, C, K, act, f32):
    w = rng.integers(-127, 128, (K, C, 1, 1)).astype(np.int8)
    ws = rng.uniform(40, 400, K).astype(np.float32) * np.float32(np.sqrt(C))
    return hip.conv(wq=w, scale_in=host_scale_in(ws, 31.0), bias=rng.normal(0, 0.4, K).astype(np.float32), in_scale=31.0,
                    out_scale=None if f32 else [23.0], act=act, act_p0=0.1, out_kind=capi.OUT_F32 if f32 else capi.OUT_I8,
                    out_round=capi.ROUND_SSE)


def one_and_two(hip, a, b, x, n, h, w, form, rng, K):
    """(the launch's results, the results of the layers one by one)"""
    blob = lambda: hip.to_device(rng.normal(0, 2, n * K * h * w).astype(np.float32))
    new = lambda dtype: hip.empty(n * K * h * w, dtype).fill_(77)
    then = lambda q: b.forward(q, capi.I8_P8, n, h, w, hip._packed_out(b))
    if form == "i8":
        return (hip.conv_pair(a, b, x, n, h, w),), (then(a.forward(x, capi.I8_P8, n, h, w, capi.I8_P8)),)
    got = []
    want = []
    for odd, layout in ((0, capi.F32_P8), (1, capi.F32_P4)):
        other, lo = blob(), new(np.float32)
        got += [hip.conv_pair(a, b, x, n, h, w, first_half=lo, other=other, other_layout=layout, other_odd=odd, q_scale=19.0, q_round_mode=capi.ROUND_SSE), lo]
        t = a.forward_shuffle(x, n, h, w, other, layout, bool(odd), False, 19.0)
        want += [then(t[3]), t[0]]
    return got, want


def test_which_are_one_launch(hip):
    rng = np.random.default_rng(5)
    for C, n, h, one in ((88, 1, 13, 1), (88, 16, 52, 1), (176, 1, 13, 2), (176, 16, 13, 1), (352, 16, 13, 2), (352, 16, 26, 1), (48, 16, 26, 1),
                         (48, 16, 52, 2)):
        a, b = layer(hip, rng, C, C, 2, False), layer(hip, rng, C, C, 2, False)
        assert hip.conv_pair_launches(a, b, n, h, h) == one, (C, n, h)
    # channels that one workgroup would walk for all the others, first layers of two pairs on large batches
    for C, K, K2, n, h, one in ((64, 128, 1280, 1, 7, 2), (64, 128, 1280, 16, 7, 2), (128, 512, 128, 1, 14, 2), (88, 88, 88, 64, 56, 1),
                                (128, 64, 128, 64, 56, 2), (128, 16, 64, 1, 14, 1), (136, 24, 40, 1, 7, 1)):
        a, b = layer(hip, rng, C, K, 2, False), layer(hip, rng, K, K2, 2, False)
        assert hip.conv_pair_launches(a, b, n, h, h) == one, (C, K, K2, n, h)


@pytest.mark.parametrize("C,K,K2,n,h,w,act0,act1", CASES)
def test_one_launch_equals_the_two_layers(hip, C, K, K2, n, h, w, act0, act1):
    rng = np.random.default_rng(C * 7 + K + w)
    x = hip.to_device(rng.integers(-127, 128, n * C * h * w).astype(np.int8))
    for form in ("i8", "shuffle"):
        a = layer(hip, rng, C, K, act0, form != "i8")
        for f32 in (False, True):
            b = layer(hip, rng, K, K2, act1, f32)
            a.set_tile(0, 0)
            r = hip.empty(n * K * h * w, np.float32)
            faster = hip.conv_pair_launches(a, b, n, h, w, **({} if form == "i8" else dict(other=r, other_layout=capi.F32_P8, first_half=r))) == 1
            for force in (0, 1, 2):  # pixel groups of a workgroup
                a.set_tile(-11 if force else 0, force)
                if not force and not faster:
                    continue
                got, want = one_and_two(hip, a, b, x, n, h, w, form, rng, K)
                hip.torch.cuda.synchronize()
                for k, (g, v) in enumerate(zip(got, want)):
                    assert hip.torch.equal(g, v), (form, f32, force, k)
            b.close()
        a.close()


def test_what_is_refused(hip):
    rng = np.random.default_rng(3)
    x = hip.empty(4 * 64 * 16, np.int8)
    a, b, odd = layer(hip, rng, 64, 64, 0, True), layer(hip, rng, 64, 64, 0, False), layer(hip, rng, 64, 60, 0, True)
    r = hip.empty(4 * 64 * 16, np.float32)
    tail = dict(other=r, other_layout=capi.F32_P8, first_half=hip.empty(4 * 64 * 16, np.float32), q_scale=1.0)
    assert hip.conv_pair_launches(a, b, 4, 4, 4, **tail) == 1 and hip.conv_pair_launches(b, b, 4, 4, 4) == 1
    for first, second, t in ((odd, b, tail), (a, b, {}), (b, a, tail), (a, b, dict(tail, other_layout=capi.F32)), (a, b, dict(tail, q_round_mode=7)),
                             (a, b, dict(tail, first_half=None))):
        with pytest.raises(capi.HipError):
            hip.conv_pair(first, second, x, 4, 4, 4, **t)
