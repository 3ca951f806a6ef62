"""Passes that a Net records and replays (Session.run and Net.eval from the third pass on): every replay gives what a pass made launch
by launch gives, with other work in between, and a net whose weights have changed is recorded anew."""
import os
import threading

import numpy as np
import pytest

from tensor_amd import hostnet, mobilenet, modelfile

pytestmark = pytest.mark.gpu

SIDE = 64


def classifier(rng, n, side=SIDE):
    layers = mobilenet.describe()
    params = mobilenet.init_weights(layers, rng)
    for l in layers:
        if l["kind"] == "conv":
            params[l["name"]].update(in_scale=20.0, top_scale=20.0 if l["int8_out"] else 1.0)
    return mobilenet.build_net(hostnet, layers, params, n, side), layers, params


class Counted:
    """What has been recorded, replayed and refused since it was made."""

    def __init__(self):
        self.start = hostnet.recording_counts()

    def __call__(self):
        return tuple(b - a for a, b in zip(self.start, hostnet.recording_counts()))


def unrecorded(net, x, out="fc", into="data"):
    return net.run(into, x, out)  # (never recorded)


@pytest.mark.parametrize("n", [1, 3])
def test_session_replays_equal_passes_by_launches(hip, n):
    rng = np.random.default_rng(n)
    net, _, _ = classifier(rng, n)
    x = rng.random((n, 3, SIDE, SIDE), dtype=np.float32)
    want = unrecorded(net, x).reshape(n, 1000)
    s = net.session("data", x, "fc")
    other = rng.random((n, 3, SIDE, SIDE), dtype=np.float32)
    busy = hip.empty(1 << 20, np.float32)
    counted = Counted()
    for i in range(8):
        s.run()
        assert counted() == ((1, i - 1, 0) if i > 1 else (0, 0, 0)), i
        if i % 2:
            unrecorded(net, other)  # takes and gives back blobs of the same sizes
            busy.zero_()
        np.testing.assert_array_equal(s.fetch((n, 1000), np.float32), want)
    s.close()
    net.close()


def test_eval_replays_on_new_inputs_and_shapes(hip):
    rng = np.random.default_rng(5)
    net, _, _ = classifier(rng, 2)
    counted = Counted()
    for i in range(10):
        n, side = ((2, SIDE), (1, SIDE), (2, 96))[i % 3 if i < 6 else 0]
        x = rng.random((n, 3, side, side), dtype=np.float32)
        np.testing.assert_array_equal(net.eval({"data": x}, "fc").reshape(n, 1000), unrecorded(net, x).reshape(n, 1000))
    # (a first pass of a shape asks for the size alone; of the others the third is recorded)
    assert counted() == (1, 3, 0)
    # a blob inside the net, a packed one
    name = next(l["name"] for l in mobilenet.describe() if l["kind"] == "add")
    for i in range(5):
        x = rng.random((1, 3, SIDE, SIDE), dtype=np.float32)
        np.testing.assert_array_equal(net.eval({"data": x}, name), unrecorded(net, x, name))
    assert counted() == (2, 5, 0)
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
            counted = Counted()
            for _ in range(5):
                s.run()
                np.testing.assert_array_equal(s.fetch((1, 1000), np.float32).reshape(-1), want)
                np.testing.assert_array_equal(net.eval({"data": x}, "fc").reshape(-1), want)
            assert counted() == (2, 5 if rnd == 0 else 6, 0), rnd  # (the first eval asks for the size alone)
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
    counted = Counted()

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
    recorded, replayed, refused = counted()
    assert recorded == 1 and 1 <= replayed <= 36 and refused == 0  # (a thread whose turn it is not launches for itself)
    net.close()


HEADS = ["conv_95", "conv_100", "conv_105", "conv_110"]


@pytest.mark.parametrize("last", HEADS)
def test_detector_with_several_results(hip, tmp_path, last):
    net = hostnet.Net()
    net.load_otter(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "nanodet-plus-m-1.5x_416_int8_fused.otter"))
    weights, _ = modelfile.synthetic_int8_weights(net.describe(), np.random.default_rng(3))
    path = tmp_path / "weights.bin"
    path.write_bytes(weights)
    net.load_weight(str(path), ncnn=True)
    x = np.random.default_rng(4).random((1, 3, 416, 416), dtype=np.float32)
    want = unrecorded(net, x, last, into="data_1")
    s = net.session("data_1", x, ",".join([h for h in HEADS if h != last] + [last]))
    counted = Counted()
    for i in range(6):
        s.run()
        np.testing.assert_array_equal(s.fetch(want.shape, want.dtype), want)
    assert counted() == (1, 4, 0)
    s.close()
    net.close()


def stack(rng, layers, C, side, kernel, n=2, int8_in=False):
    net = hostnet.Net()
    net.add_layer(type="Input", name="data", batchsize=n, channel=C, height=side, width=side)
    for i in range(layers):
        net.add_layer(type="Convolution", name="s%d" % i, out_channels=C, kernel=kernel, padding=kernel // 2,
                      int8_scale_term=102 if i < layers - 1 else 2, activation="Relu")
    net.compile()
    for i in range(layers):
        net.set_conv("s%d" % i, rng.integers(-127, 128, (C, C, kernel, kernel)).astype(np.int8), rng.normal(0, 0.1, C).astype(np.float32),
                     rng.uniform(300, 900, C).astype(np.float32), 25.0, 25.0)
    return net, "s%d" % (layers - 1)


def test_an_int8_input(hip):
    rng = np.random.default_rng(8)
    net, out = stack(rng, 13, 24, 9, 5)
    counted = Counted()
    x = rng.integers(-127, 128, (2, 24, 9, 9)).astype(np.int8)
    want = unrecorded(net, x, out)
    assert len(np.unique(want)) > 100
    s = net.session("data", x, out)
    for i in range(6):
        s.run()
        y = rng.integers(-127, 128, x.shape).astype(np.int8)
        np.testing.assert_array_equal(net.eval({"data": y}, out), unrecorded(net, y, out))
        s.run()
    assert s.fetch((want.size,), np.float32).size == want.size and counted()[0] == 2 and counted()[1] >= 10
    np.testing.assert_array_equal(net.eval({"data": x}, out), want)
    s.close()
    net.close()


def test_a_net_with_a_chain_goes_on_without_a_recording(hip):
    rng = np.random.default_rng(9)
    tiles = hip.conv_chain_set_min_tiles(0)
    try:
        net, out = stack(rng, 14, 64, 14, 3)
        chains = hostnet.chain_forward_count()
        counted = Counted()
        x = rng.random((2, 64, 14, 14), dtype=np.float32)
        want = unrecorded(net, x, out)
        assert hostnet.chain_forward_count() > chains and len(np.unique(want)) > 100
        s = net.session("data", x, out)
        for i in range(6):
            s.run()
            y = rng.random(x.shape, dtype=np.float32)
            np.testing.assert_array_equal(net.eval({"data": y}, out), unrecorded(net, y, out))
            np.testing.assert_array_equal(net.eval({"data": x}, out), want)
        recorded, replayed, refused = counted()
        assert (recorded, replayed) == (0, 0) and refused >= 1
        s.close()
        net.close()
    finally:
        hip.conv_chain_set_min_tiles(tiles)


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
