"""otter_hip_conv_dwpw_forward: a depthwise layer, the pointwise layer behind it and the one behind that in one launch. The results must be,
bit for bit, what the layers give one by one through the calls for what their ends carry."""
import ctypes

import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu

CASES = [
    # C, kernel, stride, pad, dilation, act of the depthwise layer, K, K2, N, H, W
    (88, 3, 1, 1, 1, 0, 88, 88, 2, 13, 13),       # an odd count of octets, pairs that are no multiple of the waves
    (176, 3, 2, 1, 1, 0, 176, 40, 2, 26, 26),
    (384, 3, 1, 1, 1, 3, 64, 384, 1, 14, 14),     # six reduction steps: two rounds of weights; more pairs behind than in front
    (960, 3, 1, 1, 1, 1, 160, 960, 1, 7, 7),      # the longest reduction; 49 pixels an image
    (32, 3, 1, 1, 1, 3, 16, 96, 1, 20, 31),       # half a pair: seven of eight waves begin with the second layer
    (8, 3, 1, 0, 1, 2, 8, 8, 3, 3, 3),            # one pixel an image, no padding
    (24, 3, 2, 0, 2, 2, 40, 24, 2, 9, 12),        # dilation, the window off the image's end; channels past the last ones
    (64, 3, 3, 2, 1, 2, 264, 72, 1, 11, 10),      # more padding than the window needs, a stride of three
    (128, 5, 1, 2, 1, 2, 128, 112, 2, 13, 13),
    (128, 5, 2, 2, 1, 2, 128, 128, 1, 26, 27),
    (40, 5, 1, 1, 2, 0, 24, 8, 1, 12, 9),
]


def weights(rng, K, C, k):
    return rng.integers(-127, 128, (K, C, k, k)).astype(np.int8), rng.uniform(40, 400, K).astype(np.float32) * np.float32(np.sqrt(C * k * k))


def layer(hip, rng, C, K, act, f32, half=capi.ROUND_SSE, scale=23.0, gain=1):
    w, ws = weights(rng, K, C, 1)
    return hip.conv(wq=w, scale_in=host_scale_in(ws / np.float32(gain), 31.0), bias=rng.normal(0, 0.4, K).astype(np.float32), in_scale=31.0,
                    out_scale=None if f32 else [scale], act=act, act_p0=0.1, out_kind=capi.OUT_F32 if f32 else capi.OUT_I8, out_round=half)


def depthwise(hip, rng, C, k, stride, pad, dil, act, half=capi.ROUND_SSE, scale=37.0):
    w, ws = weights(rng, C, 1, k)
    return hip.conv(wq=w, scale_in=host_scale_in(ws, 29.0), bias=rng.normal(0, 0.4, C).astype(np.float32), in_scale=29.0, out_scale=[scale], act=act,
                    act_p0=0.2, groups=C, stride=(stride, stride), pad=(pad, pad), dil=(dil, dil), out_kind=capi.OUT_I8, out_round=half)


def forms(k, last):
    """(name, fields of the end beside the blobs) that run with this window, without and with a layer behind the pointwise one"""
    shuffles = [("shuffle", dict(odd=odd, layout=layout)) for odd, layout in ((0, capi.F32_P8), (1, capi.F32_P4))]
    if last:
        return [("i8", {})] + ([("sum", {}), ("f32", {}), ("wanted", {})] + shuffles if k == 3 else [])
    return [("i8", {}), ("f32", {}), ("twin", {}), ("sum", {}), ("parts", {})] + (shuffles + [("joined", dict(odd=1, layout=capi.F32_P8))] if k == 3 else [])


def one_and_two(hip, rng, form, how, dw, pw, nx, x, n, h, w):
    """(the launch's results, those of the layers one by one)"""
    K, (oh, ow) = pw.K, dw.out_hw(h, w)
    count = n * K * oh * ow
    blob = lambda c=K: hip.to_device(rng.normal(0, 2, n * c * oh * ow).astype(np.float32))
    new = lambda dtype, k=1: hip.empty(k * count, dtype).fill_(77)
    q = dict(q_scale=19.0, q_round_mode=capi.ROUND_EXACT if K % 16 else capi.ROUND_SSE)
    run = lambda **end: hip.conv_dwpw(dw, pw, x, n, h, w, next=nx, **end)
    force = dw.force
    dw.set_tile(0, 0)
    mid = dw.forward(x, capi.I8_P8, n, h, w, capi.I8_P8)
    dw.set_tile(*force)
    then = lambda t: [nx.forward(t, capi.I8_P8, n, oh, ow, hip._packed_out(nx))] if nx else []
    if form == "i8":
        t = pw.forward(mid, capi.I8_P8, n, oh, ow, capi.I8_P8)
        return [run()], then(t) if nx else [t]
    if form in ("f32", "twin", "wanted"):
        f, t = pw.forward_twin(mid, capi.I8_P8, n, oh, ow, q["q_scale"], q["q_round_mode"])
        if nx:
            s = new(np.float32) if form == "wanted" else None
            return [run(sum=s, **q)] + [s] * (form == "wanted"), then(t) + [f] * (form == "wanted")
        if form == "f32":
            return [run()], [f]
        o, only = new(np.int8), new(np.int8)
        got = run(out_q=o, **q)
        hip.conv_dwpw(dw, pw, x, n, h, w, wants_out=False, out_q=only, **q)
        return [got, o, only], [f, t, t]
    if form == "sum":
        r = blob()
        f, t = pw.forward_residual(mid, capi.I8_P8, n, oh, ow, r, q["q_scale"], q["q_round_mode"])
        if nx:
            s = new(np.float32)
            return [run(residual=r, sum=s, **q), s], then(t) + [f]
        o = new(np.int8)
        return [run(residual=r, out_q=o, **q), o, run(residual=r)], [f, t, f]
    if form == "parts":
        c0 = max(8, K // 16 * 8) if K > 8 else 0
        if not c0:
            return [], []
        a, b, o = blob(c0), blob(K - c0), new(np.int8)
        f, t = pw.forward_residual_concat(mid, n, oh, ow, a, capi.F32_P4, c0, b, capi.F32_P8, **q)
        return [run(residual=a, residual1=b, part0_channels=c0, part0_layout=capi.F32_P4, part1_layout=capi.F32_P8, out_q=o, **q), o], [f, t]
    other = blob()
    end = dict(other=other, other_layout=how["layout"], other_odd=how["odd"], **q)
    t = pw.forward_shuffle(mid, n, oh, ow, other, how["layout"], bool(how["odd"]), form == "joined", q["q_scale"], q["q_round_mode"])
    if form == "joined":
        f, o = new(np.float32, 2), new(np.int8, 2)
        hip.conv_dwpw(dw, pw, x, n, h, w, wants_out=False, joined=1, first_half=f, first_half_q=o, **end)
        return [f, o], [t[0], t[2]]
    lo, p4 = new(np.float32), new(np.float32)

    def float8(t):  # what is Float4, as Float8
        return t.view(n, K // 8, 2, oh * ow, 4).permute(0, 1, 3, 2, 4).reshape(-1)
    if nx:
        return [run(first_half=lo, **end), lo, run(first_half=p4, first_float4=1, **end), float8(p4)], (then(t[3]) + [t[0]]) * 2
    hi, lq, hq = new(np.float32), new(np.int8), new(np.int8)
    hip.conv_dwpw(dw, pw, x, n, h, w, wants_out=False, first_half=lo, second_half=hi, first_half_q=lq, second_half_q=hq, **end)
    hip.conv_dwpw(dw, pw, x, n, h, w, wants_out=False, first_half=p4, first_float4=1, second_half_q=hq, **end)
    return [lo, hi, lq, hq, float8(p4)], list(t) + [t[0]]


@pytest.mark.parametrize("C,k,stride,pad,dil,act,K,K2,n,h,w", CASES)
def test_one_launch_equals_the_layers(hip, C, k, stride, pad, dil, act, K, K2, n, h, w):
    rng = np.random.default_rng(C * 7 + K + w)
    x = hip.to_device(rng.integers(-127, 128, n * C * h * w).astype(np.int8))
    dw = depthwise(hip, rng, C, k, stride, pad, dil, act, capi.ROUND_EXACT if K % 16 else capi.ROUND_SSE)
    for last in (None, "i8", "nonneg", "f32"):
        nx = layer(hip, rng, K, K2, {"nonneg": 3, "i8": 2, "f32": 1, None: 0}[last], last == "f32") if last else None
        for form, how in forms(k, last):
            pw = layer(hip, rng, C, K, 2 if form != "sum" else 0, form != "i8")
            for groups in (1, 2, 4, 8, 17, 18, 20):  # of 16 pixels, + 16 with four waves
                if 16 * (groups & 15) * (C + 160 + (K + 160 if nx else 0)) > 60000:
                    continue
                dw.force = (-12, groups)
                dw.set_tile(-12, groups)
                got, want = one_and_two(hip, rng, form, how, dw, pw, nx, x, n, h, w)
                hip.torch.cuda.synchronize()
                assert len(got) == len(want)
                for i, (g, v) in enumerate(zip(got, want)):
                    assert hip.torch.equal(g, v), (last, form, how, groups, i)
            pw.close()


def staged_lds(C, k, pad, dil, K, K2, H, W, groups):
    """Bytes of LDS of a plan with staged pixels: rows of a tile's pixels, what is staged (or the second layer's rows), the constants."""
    up = lambda v, to: -(-v // to) * to
    pixels = 16 * groups
    places = pixels + (k - 1) * (dil * W + dil) + (max(0, (pixels + H * W - 2) // (H * W)) if H * W % 2 else 0)
    units = up(1 + places, 2) // 2 + 1
    lanes = min(64, 1 << (units - 1).bit_length())
    octets, pitch = up(up(C // 8, 2), 64 // lanes), 2 * units if units > 64 else 2 * lanes
    weights = up(up(C // 8, 2) // 2 * 256 * (2 if k == 3 else 4), 1024)
    row = lambda c: up(c, 64) + 16
    return (pixels * row(C) + max(8 * octets * pitch + weights, pixels * row(K) if K2 else 0) + 256 * (up(K, 32) + up(K2, 32)) // 32
            + 128 * (up(C // 8, 2) // 2))


@pytest.mark.parametrize("C,k,pad,dil,act,K,K2,N,H,W", [
    (88, 3, 1, 1, 0, 88, 88, 3, 13, 13),     # an odd count of octets, images of an odd count of pixels that begin inside a tile
    (16, 3, 1, 1, 3, 24, 16, 9, 3, 3),       # several images in a tile, octets that share a copy
    (8, 3, 1, 1, 2, 8, 8, 21, 1, 1),         # one pixel an image
    (72, 3, 2, 2, 2, 40, 24, 2, 12, 9),      # dilation
    (32, 3, 1, 1, 3, 16, 96, 1, 7, 112),     # an octet takes several copies
    (256, 3, 1, 1, 1, 64, 128, 1, 14, 14),
    (128, 5, 2, 1, 2, 128, 112, 2, 13, 13),
    (40, 5, 2, 1, 0, 24, 8, 1, 26, 40),
    (24, 5, 4, 2, 3, 24, 8, 3, 5, 7),
])
def test_staged_pixels(hip, C, k, pad, dil, act, K, K2, N, H, W):
    """The plans (+ 32) that copy the windows' pixels into LDS first."""
    rng = np.random.default_rng(C + K + W)
    x = hip.to_device(rng.integers(-127, 128, N * C * H * W).astype(np.int8))
    dw = depthwise(hip, rng, C, k, 1, pad, dil, act)
    for last in (None, "nonneg"):
        nx = layer(hip, rng, K, K2, 3, False) if last else None
        for form, how in forms(k, last):
            pw = layer(hip, rng, C, K, 2 if form != "sum" else 0, form != "i8")
            for plan in (33, 34, 36, 40, 49, 50, 52):
                dw.force = (-12, plan)
                dw.set_tile(-12, plan)
                if staged_lds(C, k, pad, dil, K, K2 if nx else 0, H, W, plan & 15) > 65536:
                    assert C > 16  # (the smaller ones run every plan)
                    with pytest.raises(capi.HipError):
                        one_and_two(hip, rng, form, how, dw, pw, nx, x, N, H, W)
                    continue
                got, want = one_and_two(hip, rng, form, how, dw, pw, nx, x, N, H, W)
                assert len(got) == len(want)
                for i, (g, v) in enumerate(zip(got, want)):
                    assert hip.torch.equal(g, v), (last, form, how, plan, i)


@pytest.mark.parametrize("scale,next_scale", [(9.0, 23.0), (37.0, 9.0), (21.0, 9.0)])  # clip: 6 * 9 and 6 * 21 are below 127
@pytest.mark.parametrize("C,k,stride,K,K2,n,h,w", [(88, 3, 1, 88, 88, 2, 13, 13), (40, 3, 2, 24, 40, 2, 17, 12), (128, 5, 1, 128, 112, 1, 13, 13)])
def test_clamps_below_the_bytes_end(hip, C, k, stride, K, K2, n, h, w, scale, next_scale):
    """Clip with an upper clamp below 127, in the depthwise layer, the last one or both."""
    rng = np.random.default_rng(C + k)
    x = hip.to_device(rng.integers(-127, 128, n * C * h * w).astype(np.int8))
    dw = depthwise(hip, rng, C, k, stride, k // 2, 1, 3, scale=scale)
    mid = dw.forward(x, capi.I8_P8, n, h, w, capi.I8_P8)
    assert mid.max() == min(127, 6 * scale) and mid.min() == 0
    for last in (False, True):
        nx = layer(hip, rng, K, K2, 3, False, scale=next_scale, gain=16) if last else None
        for form, how in forms(k, last):
            pw = layer(hip, rng, C, K, 2 if form != "sum" else 0, form != "i8")
            for plan in (2, 18) + ((34, 50) if stride == 1 else ()):
                dw.force = (-12, plan)
                dw.set_tile(-12, plan)
                got, want = one_and_two(hip, rng, form, how, dw, pw, nx, x, n, h, w)
                assert not last or want[0].max() == min(127, 6 * next_scale)
                for i, (g, v) in enumerate(zip(got, want)):
                    assert hip.torch.equal(g, v), (last, form, how, plan, i)


def test_a_blob_at_an_odd_address(hip):
    """An input that is not on eight bytes is not copied in pairs of pixels: refused where that is forced, another plan otherwise."""
    rng = np.random.default_rng(9)
    n, C, side = 2, 88, 13
    values = rng.integers(-127, 128, n * C * side * side).astype(np.int8)
    dw, pw = depthwise(hip, rng, C, 3, 1, 1, 1, 0), layer(hip, rng, C, 88, 2, False)
    base = hip.empty(values.size + 16, np.int8)
    base[4:4 + values.size] = hip.to_device(values)
    dw.set_tile(-12, 0)
    want = hip.conv_dwpw(dw, pw, hip.to_device(values), n, side, side)
    assert hip.torch.equal(hip.conv_dwpw(dw, pw, base[4:4 + values.size], n, side, side), want)
    dw.set_tile(-12, 34)
    with pytest.raises(capi.HipError):
        hip.conv_dwpw(dw, pw, base[4:4 + values.size], n, side, side)


@pytest.mark.parametrize("C,k,stride,K,K2,n,side,form,ratio", [
    # drawn layers, the launch's time over that of the layers one by one where the rule was measured
    (32, 3, 1, 32, 32, 6, 88, "shuffle", 0.60), (72, 3, 1, 72, 24, 9, 13, "sum", 0.61), (48, 3, 1, 16, 96, 7, 19, "f32", 0.62),
    (120, 3, 1, 32, 0, 6, 24, "i8", 0.71), (128, 5, 1, 128, 112, 16, 13, "i8", 0.75),
    (952, 3, 2, 952, 0, 2, 8, "f32", 3.47), (600, 5, 2, 600, 0, 1, 10, "i8", 2.99), (848, 3, 1, 848, 848, 3, 10, "i8", 2.56),
    # many channels and many pixels, where the models are too kind to the launch
    (384, 3, 1, 32, 0, 29, 76, "f32", 1.3), (144, 3, 1, 32, 0, 49, 80, "f32", 1.3),  # ten million values and more, in a block with its expand layer
    # 5x5 in a last round of workgroups that few of them fill; more bytes than the caches hold
    (136, 5, 1, 136, 136, 4, 65, "i8", 1.33), (256, 5, 1, 24, 112, 43, 20, "i8", 1.31), (512, 5, 2, 512, 0, 42, 40, "sum", 1.39), (168, 5, 1, 168, 168, 8, 48, "i8", 1.33),
    (600, 3, 1, 600, 0, 12, 28, "f32", 1.22), (520, 3, 1, 520, 32, 11, 81, "shuffle", 1.23), (48, 5, 1, 416, 0, 50, 32, "sum", 1.34),
    (664, 3, 1, 664, 32, 7, 49, "f32", 1.50), (696, 3, 1, 696, 120, 4, 75, "i8", 1.47), (904, 3, 2, 904, 904, 3, 78, "f32", 1.19),
])
def test_the_launch_is_taken_where_it_is_faster(hip, C, k, stride, K, K2, n, side, form, ratio):
    """Which way the rule decides by itself, and the result of the plan that it chooses."""
    rng = np.random.default_rng(C + side)
    dw, pw = depthwise(hip, rng, C, k, stride, k // 2, 1, 0), layer(hip, rng, C, K, 0, form != "i8")
    nx = layer(hip, rng, K, K2, 2, False) if K2 else None
    x = hip.to_device(rng.integers(-127, 128, n * C * side * side, dtype=np.int8))
    some = hip.empty(4, np.float32)  # (of the pointers it is only asked which are null)
    end = dict(dict(q_scale=19.0, q_round_mode=1) if nx and form != "i8" else {}, **{"shuffle": dict(other=some, other_layout=capi.F32_P8, first_half=some),
                                                                                     "sum": dict(residual=some)}.get(form, {}))
    assert hip.conv_dwpw_launches(dw, pw, n, side, side, next=nx, **end) == (1 if ratio < 1 else 2)
    if ratio < 1:
        dw.force = (0, 0)
        got, want = one_and_two(hip, rng, form, dict(odd=0, layout=capi.F32_P8), dw, pw, nx, x, n, side, side)
        for g, v in zip(got, want):
            assert hip.torch.equal(g, v)


@pytest.mark.parametrize("n", [16, 17])  # 2^30 bytes of int8 result, and 64 MiB more
def test_an_int8_result_of_a_gigabyte(hip, n):
    C, K, h, w = 64, 1024, 256, 256
    rng = np.random.default_rng(n)
    x = hip.to_device(rng.integers(-127, 128, n * C * h * w, dtype=np.int8))
    dw, pw = depthwise(hip, rng, C, 3, 1, 1, 1, 0), layer(hip, rng, C, K, 2, False)
    want = pw.forward(dw.forward(x, capi.I8_P8, n, h, w, capi.I8_P8), capi.I8_P8, n, h, w, capi.I8_P8)
    dw.set_tile(-12, 0)
    unwritten = hip.empty(n * K * h * w, np.int8).fill_(77)  # (the memory that the result is given next)
    del unwritten
    assert hip.torch.equal(hip.conv_dwpw(dw, pw, x, n, h, w), want)


def test_an_empty_batch(hip):
    rng = np.random.default_rng(1)
    dw, pw, buf, end = depthwise(hip, rng, 64, 3, 1, 1, 1, 0), layer(hip, rng, 64, 64, 0, False), hip.empty(64, np.int8).fill_(5), hip._end({})
    call = lambda n, h: hip.lib.otter_hip_conv_dwpw_forward(dw.h, pw.h, hip.ptr(buf), n, h, 6, ctypes.byref(end), hip.ptr(buf), capi.I8_P8, hip.stream())
    assert call(0, 6) == 0 and (buf == 5).all()
    assert call(0, 0) < 0 and call(-1, 6) < 0


def test_what_is_refused(hip):
    rng = np.random.default_rng(3)
    n, h, w = 2, 6, 6
    x = hip.empty(n * 64 * h * w, np.int8)
    dw = depthwise(hip, rng, 64, 3, 1, 1, 1, 0)
    dw.set_tile(-12, 0)
    i8, f32, odd, clipped = (layer(hip, rng, 64, K, act, f) for K, act, f in ((64, 0, False), (64, 0, True), (60, 0, True), (64, 1, False)))
    r, b = hip.empty(n * 64 * h * w, np.float32), hip.empty(n * 64 * h * w, np.int8)
    other = dict(other=r, other_layout=capi.F32_P8, first_half=r.clone(), q_scale=1.0)
    assert hip.conv_dwpw_launches(dw, i8, n, h, w) == 1 and hip.conv_dwpw_launches(dw, f32, n, h, w, next=i8, **other) == 1
    assert hip.conv_dwpw_launches(dw, clipped, n, h, w) == 2  # (its clamp is not among this launch's ends)
    assert hip.conv_dwpw_launches(dw, odd, n, h, w) == 1      # (Float4 alone)
    for first, second, end in ((i8, i8, {}), (dw, dw, {}), (dw, i8, dict(residual=r)), (dw, i8, other), (dw, i8, dict(out_q=b)), (dw, odd, dict(out_q=b, q_scale=1.0)),
                               (dw, odd, dict(next=i8)), (dw, f32, dict(next=i8, out_q=b)), (dw, f32, dict(sum=r)), (dw, f32, dict(residual1=r)),
                               (dw, f32, dict(next=i8, q_round_mode=9)), (dw, f32, dict(other, residual=r)), (dw, f32, dict(other, first_half=None, next=i8)),
                               (dw, f32, dict(other, joined=1, second_half=r)), (dw, f32, dict(other, joined=1, first_float4=1)), (dw, f32, dict(other, other_layout=capi.F32)), (dw, clipped, {}),
                               (dw, f32, dict(residual=r, residual1=r, part0_channels=60, part0_layout=capi.F32_P8, part1_layout=capi.F32_P8))):
        with pytest.raises(capi.HipError):
            hip.conv_dwpw(first, second, x, n, h, w, **end)
