"""Copies through the library's staging buffers and through pinned memory: byte for byte, at the edges of their pieces."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@pytest.mark.parametrize("count", [1, 15, 4000, MIB - 1, MIB, MIB + 1, 3 * MIB + 5, 20 * MIB])
def test_upload_and_download(hip, count):
    torch, lib = hip.torch, hip.lib
    failures = []

    def worker(seed):
        src = np.random.default_rng(seed).integers(0, 256, count, dtype=np.uint8)
        dev = torch.zeros(count + 64, dtype=torch.uint8, device="cuda")
        back = np.zeros(count + 1, np.uint8)
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(3):
                hip._check(lib.otter_hip_upload(hip.ptr(dev), C.c_void_p(src.ctypes.data), C.c_size_t(count), hip.stream()))
                dev[:count] ^= 255  # a launch on the copy's stream sees all of it
                back[:] = 7
                hip._check(lib.otter_hip_download(C.c_void_p(back.ctypes.data), hip.ptr(dev), C.c_size_t(count), hip.stream()))
                if not ((back[:count] == src ^ 255).all() and back[count] == 7 and int(dev[count:].sum()) == 0):
                    failures.append(seed)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=worker, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures


@pytest.mark.parametrize("count", [1, 16, 31, 256 * 16, 256 * 256 * 16 + 3, 2 * MIB + 7])
def test_copy_from_pinned_memory(hip, count):
    lib, pin = hip.lib, C.c_void_p()
    hip._check(lib.otter_hip_host_malloc(C.byref(pin), C.c_size_t(count)))
    src = np.random.default_rng(count).integers(0, 256, count, dtype=np.uint8)
    C.memmove(pin, src.ctypes.data, count)
    dev = hip.torch.zeros(count + 64, dtype=hip.torch.uint8, device="cuda")
    hip._check(lib.otter_hip_copy(hip.ptr(dev), pin, C.c_size_t(count), hip.stream()))
    got = dev.cpu().numpy()
    assert (got[:count] == src).all() and not got[count:].any()
    hip._check(lib.otter_hip_host_free(pin))
