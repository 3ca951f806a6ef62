"""CPU: the pinned buffers that host inputs of the Net pass through, over a stand-in for the few entry points of the GPU library
that a pass over an Input layer alone makes."""
import subprocess
import sys

from tensor_amd import hostnet

FAKE = r"""
#include <stdlib.h>
#include <string.h>
static int fail_copies, allocated, held;
int otter_hip_init(int d) { return 0; }
const char* otter_hip_last_error(void) { return "a copy that fails"; }
int otter_hip_malloc(void** p, size_t n) { *p = malloc(n); return 0; }
int otter_hip_free(void* p) { free(p); return 0; }
int otter_hip_host_malloc(void** p, size_t n) { *p = malloc(n); ++allocated; ++held; return 0; }
int otter_hip_host_free(void* p) { free(p); --held; return 0; }
int otter_hip_copy(void* d, const void* s, size_t n, void* stream) {
    if (fail_copies > 0) { --fail_copies; return -3; }
    memcpy(d, s, n);
    return 0;
}
int otter_hip_download(void* d, const void* s, size_t n, void* stream) { memcpy(d, s, n); return 0; }
int otter_hip_stream_synchronize(void* stream) { return 0; }
void fake_fail(int n) { fail_copies = n; }
int fake_allocated(void) { return allocated; }
int fake_held(void) { return held; }
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
