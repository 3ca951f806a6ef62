"""CPU: what the Net takes over the bus and when, and the pinned buffers that its host inputs pass through, over a stand-in for
the few entry points of the GPU library that an Input and an InnerProduct layer need."""
import subprocess
import sys

from tensor_amd import hostnet

FAKE = r"""
#include <stdlib.h>
#include <string.h>
static int fail_copies, allocated, uploads;
int otter_hip_init(int d) { return 0; }
const char* otter_hip_last_error(void) { return "a copy that fails"; }
int otter_hip_malloc(void** p, size_t n) { *p = malloc(n); return 0; }
int otter_hip_free(void* p) { free(p); return 0; }
int otter_hip_host_malloc(void** p, size_t n) { *p = malloc(n); ++allocated; return 0; }
int otter_hip_host_free(void* p) { free(p); return 0; }
int otter_hip_copy(void* d, const void* s, size_t n, void* stream) {
    if (fail_copies > 0) { --fail_copies; return -3; }
    memcpy(d, s, n);
    return 0;
}
int otter_hip_upload(void* d, const void* s, size_t n, void* stream) { ++uploads; memcpy(d, s, n); return 0; }
int otter_hip_inner_product(const float* x, int n, int in, const float* w, const float* b, int out, float* y, void* stream) {
    for (int i = 0; i < n * out; ++i) {
        y[i] = b ? b[i % out] : 0;
        for (int k = 0; k < in; ++k) y[i] += x[i / out * in + k] * w[i % out * in + k];
    }
    return 0;
}
int otter_hip_download(void* d, const void* s, size_t n, void* stream) { memcpy(d, s, n); return 0; }
int otter_hip_stream_synchronize(void* stream) { return 0; }
void fake_fail(int n) { fail_copies = n; }
int fake_allocated(void) { return allocated; }
int fake_uploads(void) { return uploads; }
"""

SCRIPT = r"""
import ctypes as C, sys
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # (in front of the library that the host layer names)
from tensor_amd import hostnet

def net(h, w):
    n = hostnet.Net()
    n.add_layer(type="Input", name="data", batchsize=1, channel=3, height=h, width=w)
    n.compile()
    return n
"""


def run(tmp_path, script):
    c, so = tmp_path / "fake.c", str(tmp_path / "libfake.so")
    c.write_text(FAKE)
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", str(c), "-o", so])
    r = subprocess.run([sys.executable, "-c", SCRIPT + script, so], capture_output=True, text=True, timeout=60,
                       cwd=hostnet.HERE + "/..")
    assert r.returncode == 0, r.stdout + r.stderr


def test_an_upload_that_fails_gives_its_buffer_back(tmp_path):
    run(tmp_path, r"""
n = net(200, 700)  # 1.6 MB: more than one piece
x = np.random.default_rng(0).random((1, 3, 200, 700), dtype=np.float32)
for k in range(5):
    fake.fake_fail(1)
    try:
        n.eval({"data": x}, "data")
        raise SystemExit("no error")
    except hostnet.HostError:
        pass
    assert (n.eval({"data": x}, "data") == x).all()
assert fake.fake_allocated() == 1, fake.fake_allocated()
""")


def test_inner_product_weights_cross_when_they_are_set(tmp_path):
    run(tmp_path, r"""
n = hostnet.Net()
n.add_layer(type="Input", name="data", batchsize=1, channel=3, height=2, width=2)
n.add_layer(type="InnerProduct", name="fc", out_features=5)
n.compile()
rng = np.random.default_rng(1)
for k in range(2):  # set once, and again
    w, b = rng.integers(-3, 4, (5, 12)).astype(np.float32), rng.integers(-3, 4, 5).astype(np.float32)
    n.set_inner_product("fc", w, b)
    before = fake.fake_uploads()
    assert before == 2 * (k + 1), before
    x = rng.integers(-3, 4, (1, 3, 2, 2)).astype(np.float32)
    assert (n.eval({"data": x}, "fc").ravel() == x.ravel() @ w.T + b).all()
    assert fake.fake_uploads() == before
""")


def test_an_input_of_another_size_reuses_a_buffer_that_holds_it(tmp_path):
    run(tmp_path, r"""
rng = np.random.default_rng(2)
n = net(40, 40)
for h, w, new in ((40, 40, 1), (40, 39, 1), (20, 40, 1), (40, 40, 1), (20, 39, 2), (40, 40, 2), (41, 40, 3), (40, 40, 3)):
    x = rng.random((1, 3, h, w), dtype=np.float32)
    assert (n.eval({"data": x}, "data") == x).all()
    assert fake.fake_allocated() == new, (h, w, fake.fake_allocated())
""")
