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
