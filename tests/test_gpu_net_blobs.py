"""Whatever launches the Net groups its layers into and whichever fp32 blobs it leaves out, a blob that is asked for by name is
what the layers give one at a time."""
import os

import numpy as np
import pytest

from tensor_amd import hostnet, modelfile

pytestmark = pytest.mark.gpu

NANODET = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "nanodet-plus-m-1.5x_416_int8_fused.otter")


@pytest.mark.parametrize("lightmode", [True, False])
def test_detector_blobs_by_name(tmp_path, lightmode):
    rng = np.random.default_rng(5)
    net = hostnet.Net(lightmode=lightmode)
    net.load_otter(NANODET)
    layers = net.describe()
    blob, _ = modelfile.synthetic_int8_weights(layers, rng)
    path = str(tmp_path / "weights.bin")
    with open(path, "wb") as f:
        f.write(blob)
    net.load_weight(path, ncnn=True)
    x = rng.random((2, 3, 416, 416), dtype=np.float32)
    blobs, names = {"data_1": x}, []
    for kind, name, bottoms, tops, _conv, _shape in layers:  # one layer at a time: its inputs are set, nothing to group
        if kind == "Split":
            for t in tops:
                blobs[t] = blobs[bottoms[0]]
        elif kind not in ("Input", "NanodetPlusDetectionOutput"):
            blobs[tops[0]] = net.eval({b: blobs[b] for b in bottoms}, tops[0])
        names += [t for t in tops if kind not in ("Input", "NanodetPlusDetectionOutput")]
    assert len(names) > 180
    for name in names:
        want = blobs[name]
        np.testing.assert_array_equal(net.eval({"data_1": x}, name), want, err_msg=name)  # this blob alone
        np.testing.assert_array_equal(net.run("data_1", x, name), want, err_msg=name)     # any blob may follow
    # two blobs of one pass (a light pass frees what is in the middle: there it comes first)
    for name in ("concat_20", "crop_10", "shuffle_4", "shortcut_1"):
        order = [name, "conv_95"] if lightmode else ["conv_95", name]
        if name not in blobs:
            continue
        s = net.session("data_1", x, ",".join(order))
        for _ in range(2):
            s.run()
        want = blobs[order[1]]
        np.testing.assert_array_equal(s.fetch(want.shape, want.dtype), want, err_msg=name)
        s.close()
    net.close()


def test_a_result_that_changes_its_size_or_type(oracle):
    """The same call on the same Net, whose result grows and shrinks between calls: a layer with an int8 result that runs as its
    fp32 twin for a while, and one whose output scale is set again."""
    rng = np.random.default_rng(9)
    x = rng.uniform(-1, 1, (2, 16, 9, 11)).astype(np.float32)
    wf = rng.normal(0, 0.1, (24, 16, 3, 3)).astype(np.float32)
    ws = (np.float32(127) / np.abs(wf).reshape(24, -1).max(axis=1)).astype(np.float32)
    wq = np.round(wf * ws[:, None, None, None]).astype(np.int8)
    bias = rng.normal(0, 0.1, 24).astype(np.float32)
    in_scale = np.float32(127)
    net = hostnet.Net()
    net.add_layer(type="Input", name="data", batchsize=2, channel=16, height=9, width=11)
    net.add_layer(type="Convolution", name="conv", out_channels=24, kernel=3, padding=1, int8_scale_term=102, activation="Relu")
    net.compile()

    def want(int8_out, top):
        return oracle.conv_layer_forward(x, wq, ws, in_scale, pad=(1, 1), bias=bias, top_scale=np.float32(top), int8_out=int8_out, act_type=1)

    for top in (20.0, 35.0):
        net.set_conv("conv", wq, bias, ws, in_scale, top)
        for _ in range(2):
            for probe in (False, True):
                net.conv_fp32_probe("conv", probe)
                for _ in range(2):
                    got = net.eval({"data": x}, "conv")
                    assert got.dtype == (np.float32 if probe else np.int8) and got.flags.owndata
                    np.testing.assert_array_equal(got, want(not probe, top))
        net.conv_fp32_probe("conv", False)
    with pytest.raises(hostnet.HostError):
        net.eval({"data": x}, "no such blob")
    np.testing.assert_array_equal(net.eval({"data": x}, "conv"), want(True, 35.0))
    net.close()
