"""CPU: otter_hip_upload / otter_hip_download and their staging buffers on several GPUs, over a stand-in for the HIP runtime
(fake_hip.cpp) whose copies happen only when somebody waits for them."""
import os
import subprocess
import sys

import pytest

from tensor_amd import capi

HERE = os.path.dirname(os.path.abspath(__file__))

SCRIPT = r"""
import ctypes as C, sys
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # (in front of the runtime that the library names)
lib = C.CDLL(sys.argv[2])
lib.otter_hip_last_error.restype = C.c_char_p
fake.fake_stream.restype = C.c_void_p
rng = np.random.default_rng(0)

def upload(count, stream=None):
    src, dst = rng.integers(0, 256, count, dtype=np.uint8), np.zeros(count, np.uint8)
    rc = lib.otter_hip_upload(C.c_void_p(dst.ctypes.data), C.c_void_p(src.ctypes.data), C.c_size_t(count), C.c_void_p(stream))
    return rc, src, dst

def good(rc, src, dst, stream=None):
    assert rc == 0, lib.otter_hip_last_error()
    back = np.zeros(src.size, np.uint8)
    assert lib.otter_hip_download(C.c_void_p(back.ctypes.data), C.c_void_p(dst.ctypes.data), C.c_size_t(src.size), C.c_void_p(stream)) == 0
    assert (dst == src).all() and (back == src).all()

sizes = (5, 1 << 20, (3 << 20) + 7)
"""

CASES = {
    # the null stream means the current GPU: a buffer made for the first one is no use on the second
    "each GPU in turn": """
for device in (0, 1, 2, 1, 0):
    assert fake.hipSetDevice(device) == 0
    for n in sizes:
        good(*upload(n))
""",
    # a stream names its GPU, whichever is the current one
    "streams of another GPU": """
streams = [fake.fake_stream(d) for d in (2, 0, 1)]
for _ in range(2):
    for s in streams:
        for n in sizes:
            good(*upload(n, s), s)
got = C.c_int(-1)
assert fake.hipGetDevice(C.byref(got)) == 0 and got.value == 0
""",
    # a copy whose event could not be recorded: its buffer must not be filled again while the copy is on its way
    "a record that fails": """
fake.fake_fail_records(1)
first = upload(1000)
assert first[0] != 0
second = upload(1000)
good(*second)
assert (first[2] == first[1]).all()
""",
    # a replay of the copy would read a buffer that holds something else by then
    "a stream under capture": """
s = fake.fake_stream(0)
fake.fake_capture(1)
rc, src, dst = upload(100, s)
assert rc != 0 and b"captur" in lib.otter_hip_last_error()
assert lib.otter_hip_download(C.c_void_p(dst.ctypes.data), C.c_void_p(src.ctypes.data), C.c_size_t(100), C.c_void_p(s)) != 0
good(*upload(100))
fake.fake_capture(0)
good(*upload(100, s), s)
""",
    # behind a launch of this thread on its stream one piece of the GPU's aligned memory goes by a kernel, everything else by the runtime
    "which way a download goes": """
import threading
MIB = 1 << 20
memory = np.zeros(2 * MIB, np.uint8)
memory[:] = rng.integers(0, 256, memory.size)
base = (-memory.ctypes.data) % 16
def launch(stream=None):
    a = np.zeros(64, np.uint8)
    assert lib.otter_hip_copy(C.c_void_p(memory.ctypes.data), C.c_void_p(memory.ctypes.data), C.c_size_t(16), C.c_void_p(stream)) == 0
def way(stream=None, count=4000, offset=0, of=0):
    fake.fake_memory_of(of)
    before, back = (fake.fake_copies(), fake.fake_launches()), np.zeros(count, np.uint8)
    assert lib.otter_hip_download(C.c_void_p(back.ctypes.data), C.c_void_p(memory.ctypes.data + base + offset), C.c_size_t(count), C.c_void_p(stream)) == 0
    assert (back == memory[base + offset:base + offset + count]).all()
    fake.fake_memory_of(0)
    copies, launches = fake.fake_copies() - before[0], fake.fake_launches() - before[1]
    assert copies + launches == (count + MIB - 1) // MIB and (not copies or not launches)
    return "kernel" if launches else "runtime"
a, b, other_gpu = fake.fake_stream(0), fake.fake_stream(0), fake.fake_stream(1)
for s in (None, a):
    assert way(s) == "runtime"
    launch(s)
    assert way(s) == "kernel" and way(s) == "runtime"  # (the first one has waited)
    for kw, how in ((dict(offset=4), "runtime"), (dict(offset=16), "kernel"), (dict(count=1), "kernel"), (dict(count=MIB), "kernel"), (dict(count=MIB + 1), "runtime"),
                    (dict(of=-1), "runtime"), (dict(of=1), "runtime")):
        launch(s)
        assert way(s, **kw) == how, kw
    launch(s)
    assert lib.otter_hip_stream_synchronize(C.c_void_p(s)) == 0 and way(s) == "runtime"
# a launch on one stream says nothing of another one
launch(a)
assert way(b) == "runtime" and way(None) == "runtime" and way(a) == "kernel"
launch(None)
assert lib.otter_hip_stream_synchronize(C.c_void_p(a)) == 0 and way(a) == "runtime" and way(None) == "kernel"
launch(other_gpu)
assert way(other_gpu) == "runtime"  # (memory of the current GPU alone)
# nor does another thread's
t = threading.Thread(target=launch, args=(a,))
t.start(), t.join()
assert way(a) == "runtime"
""",
    # an error that a call of the program's own has left is none of the copy's, and is still there for the program to see
    "an error of the program's own": """
data, back = rng.integers(0, 256, 4000, dtype=np.uint8), np.zeros(4000, np.uint8)
memory = np.zeros(4016, np.uint8)
memory = memory[(-memory.ctypes.data) % 16:][:4000]
memory[:] = data
args = [C.c_void_p(back.ctypes.data), C.c_void_p(memory.ctypes.data), C.c_size_t(4000), None]
assert lib.otter_hip_download(*args) == 0
for launched in (0, 1):
    if launched: assert lib.otter_hip_copy(C.c_void_p(memory.ctypes.data), C.c_void_p(memory.ctypes.data), C.c_size_t(4000), None) == 0
    fake.fake_error(9)
    back[:] = 0
    launches = fake.fake_launches()
    assert lib.otter_hip_download(*args) == 0 and (back == data).all() and fake.fake_launches() - launches == launched
    assert fake.hipGetLastError() == 9 and fake.hipGetLastError() == 0
""",
    # buffers are kept up to 16 per GPU
    "what is kept": """
for device in (0, 1):
    fake.hipSetDevice(device)
    s = fake.fake_stream(device)
    good(*upload(40 << 20, s), s)
assert 0 < fake.fake_pinned() <= 2 * 16
""",
}


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "fake_hip.cpp"), "-o", so])
    return so


@pytest.mark.parametrize("case", CASES)
def test_staging_buffers(fake, case):
    r = subprocess.run([sys.executable, "-c", SCRIPT + CASES[case], fake, capi.LIB_PATH], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
