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


@pytest.mark.parametrize("count,offset", [(1, 0), (15, 0), (16, 0), (4000, 0), (4000, 4), (256 * 16 + 7, 0), (MIB - 1, 16), (MIB, 0), (MIB + 1, 0)])
def test_download_behind_a_launch(hip, count, offset):
    """The bytes of a download behind a launch of this thread, by the copy kernel where its conditions hold (one piece of aligned memory of
    the GPU; test_staging.py sees which way each goes), and of one on an idle stream. On the null stream and on one of the program's."""
    torch, lib = hip.torch, hip.lib
    src = torch.from_numpy(np.random.default_rng(count).integers(0, 256, count + 64, dtype=np.uint8)).cuda()
    pinned = torch.zeros(count + 64, dtype=torch.uint8, pin_memory=True)
    torch.cuda.synchronize()

    def check(at):
        dev = torch.zeros(count + 64 + offset, dtype=torch.uint8, device="cuda")
        hip._check(lib.otter_hip_copy(hip.ptr(dev), hip.ptr(src), C.c_size_t(count + 64), at))  # the launch in front
        for _ in range(2):  # behind it, and on an idle stream
            back = np.full(count + 1, 7, np.uint8)
            hip._check(lib.otter_hip_download(C.c_void_p(back.ctypes.data), C.c_void_p(dev.data_ptr() + offset), C.c_size_t(count), at))
            assert (back[:count] == src.cpu().numpy()[offset:offset + count]).all() and back[count] == 7

    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            check(hip.stream())
            # pinned host memory is not the GPU's: the runtime's copy, as ever
            hip._check(lib.otter_hip_copy(hip.ptr(src), hip.ptr(src), C.c_size_t(16), hip.stream()))
            back = np.full(count, 7, np.uint8)
            hip._check(lib.otter_hip_download(C.c_void_p(back.ctypes.data), C.c_void_p(pinned.data_ptr()), C.c_size_t(count), hip.stream()))
            assert not back.any()
