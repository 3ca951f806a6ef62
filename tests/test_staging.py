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
