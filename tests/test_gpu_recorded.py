"""Passes that a Net records and replays (Session.run and Net.eval from the third pass on): every replay gives what a pass made launch
by launch gives, with other work in between, and a net whose weights have changed is recorded anew."""
import threading

import numpy as np
import pytest

from tensor_amd import capi, hostnet, mobilenet

pytestmark = pytest.mark.gpu

SIDE = 64


def classifier(rng, n, side=SIDE):
    layers = mobilenet.describe()
    params = mobilenet.init_weights(layers, rng)
    for l in layers:
        if l["kind"] == "conv":
            params[l["name"]].update(in_scale=20.0, top_scale=20.0 if l["int8_out"] else 1.0)
    return mobilenet.build_net(hostnet, layers, params, n, side), layers, params


def unrecorded(net, x, out="fc"):
    return net.run("data", x, out)  # (never recorded)


@pytest.mark.parametrize("n", [1, 3])
def test_session_replays_equal_passes_by_launches(hip, n):
    rng = np.random.default_rng(n)
    net, _, _ = classifier(rng, n)
    x = rng.random((n, 3, SIDE, SIDE), dtype=np.float32)
    want = unrecorded(net, x).reshape(n, 1000)
    s = net.session("data", x, "fc")
    other = rng.random((n, 3, SIDE, SIDE), dtype=np.float32)
    busy = hip.empty(1 << 20, np.float32)
    for i in range(8):
        s.run()
        if i % 2:
            unrecorded(net, other)  # takes and gives back blobs of the same sizes
            busy.zero_()
        np.testing.assert_array_equal(s.fetch((n, 1000), np.float32), want)
    s.close()
    net.close()


def test_eval_replays_on_new_inputs_and_shapes(hip):
    rng = np.random.default_rng(5)
    net, _, _ = classifier(rng, 2)
    for i in range(10):
        n, side = ((2, SIDE), (1, SIDE), (2, 96))[i % 3 if i < 6 else 0]
        x = rng.random((n, 3, side, side), dtype=np.float32)
        np.testing.assert_array_equal(net.eval({"data": x}, "fc").reshape(n, 1000), unrecorded(net, x).reshape(n, 1000))
    # a blob inside the net, a packed one
    name = next(l["name"] for l in mobilenet.describe() if l["kind"] == "add")
    for i in range(5):
        x = rng.random((1, 3, SIDE, SIDE), dtype=np.float32)
        np.testing.assert_array_equal(net.eval({"data": x}, name), unrecorded(net, x, name))
    net.close()


def test_new_weights_and_settings_are_recorded_anew(hip):
    rng = np.random.default_rng(6)
    net, layers, params = classifier(rng, 1)
    x = rng.random((1, 3, SIDE, SIDE), dtype=np.float32)
    s = net.session("data", x, "fc")
    stem = next(l for l in layers if l["kind"] == "conv")
    fc = next(l for l in layers if l["kind"] == "fc")
    always = hip.conv_block_set_always(0)
    try:
        for rnd in range(4):
            if rnd == 1:
                p = params[stem["name"]]
                net.set_conv(stem["name"], -p["wq"], p["bias"], p["ws"], p["in_scale"], p["top_scale"])
            if rnd == 2:
                p = params[fc["name"]]
                net.set_inner_product(fc["name"], -p["w"], p["bias"])
            if rnd == 3:
                hip.conv_block_set_always(2)
            want = unrecorded(net, x).reshape(-1)
            for _ in range(5):
                s.run()
                np.testing.assert_array_equal(s.fetch((1, 1000), np.float32).reshape(-1), want)
                np.testing.assert_array_equal(net.eval({"data": x}, "fc").reshape(-1), want)
    finally:
        hip.conv_block_set_always(always)
    s.close()
    net.close()


def test_threads_share_a_recorded_net(hip):
    rng = np.random.default_rng(7)
    net, _, _ = classifier(rng, 1)
    xs = [rng.random((1, 3, SIDE, SIDE), dtype=np.float32) for _ in range(3)]
    want = [unrecorded(net, x).reshape(-1) for x in xs]
    errors = []

    def work(i):
        try:
            for _ in range(12):
                np.testing.assert_array_equal(net.eval({"data": xs[i]}, "fc").reshape(-1), want[i])
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
        assert not t.is_alive()
    assert not errors, errors[0]
    net.close()


def test_recordings_take_launches_only(hip):
    import ctypes as C
    L, stream, rec = hip.lib, C.c_void_p(), C.c_void_p()
    a, b = hip.empty(4096, np.float32).fill_(2.0), hip.empty(4096, np.float32).fill_(0.0)
    hip.torch.cuda.synchronize()
    hip._check(L.otter_hip_record_begin(C.byref(stream)))
    hip._check(L.otter_hip_eltwise_add(hip.ptr(a), hip.ptr(a), hip.ptr(b), C.c_size_t(4096), stream))
    hip._check(L.otter_hip_record_end(stream, C.byref(rec)))
    assert float(b.sum()) == 0.0  # nothing has run yet
    for k in range(3):
        a.fill_(k)
        hip._check(L.otter_hip_record_launch(rec, hip.stream()))
        hip.torch.cuda.synchronize()
        assert bool((b == 2.0 * k).all())
    hip._check(L.otter_hip_record_destroy(rec))
    # nothing at all is no recording
    hip._check(L.otter_hip_record_begin(C.byref(stream)))
    assert L.otter_hip_record_end(stream, C.byref(rec)) != 0
