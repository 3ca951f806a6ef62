"""A layer call without a workspace of the caller's: one is made only where the chosen launches use it, with the results unchanged."""
import numpy as np
import pytest

from gpu_util import host_scale_in
from tensor_amd import capi

pytestmark = pytest.mark.gpu


def _allocations(torch, f):
    f()
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    out = f()
    return out, torch.cuda.memory_stats()["allocation.all.allocated"] - before


@pytest.mark.parametrize("C,K,k,hw,tile,made", [
    (64, 64, 3, 14, (-8, 5), 1),   # quantized by the launch itself: the output alone
    (64, 64, 3, 14, (-4, 0), 2),   # a quantize pass in front
    (20, 24, 3, 9, (0, 0), 2),     # channels padded to a multiple of 8
    (64, 64, 1, 14, (0, 0), 1),
])
def test_workspace_only_where_used(hip, C, K, k, hw, tile, made):
    rng = np.random.default_rng(C)
    conv = hip.conv(wq=rng.integers(-127, 128, (K, C, k, k)).astype(np.int8), scale_in=host_scale_in(np.full(K, 60.0, np.float32), 20.0),
                    bias=rng.normal(0, 1, K).astype(np.float32), in_scale=20.0, pad=(k // 2, k // 2), out_kind=capi.OUT_F32)
    conv.set_tile(*tile)
    layout = capi.F32_P8 if C % 8 == 0 else capi.F32_P4
    x = hip.to_device(rng.uniform(-5, 5, 2 * C * hw * hw).astype(np.float32))
    need = hip.lib.otter_hip_conv_workspace_bytes(conv.h, layout, 2, hw, hw)
    want = conv.forward(x, layout, 2, hw, hw, workspace=hip.empty(need, np.int8))
    got, count = _allocations(hip.torch, lambda: conv.forward(x, layout, 2, hw, hw))
    assert hip.torch.equal(got.view(hip.torch.int32), want.view(hip.torch.int32))
    assert count == made
    conv.close()


@pytest.mark.parametrize("C,K,n,h,w,kind,act,made", [
    (520, 264, 3, 37, 53, capi.OUT_I8, 3, 2),    # an odd count of pixels, channels that fill neither tile
    (1016, 520, 2, 40, 41, capi.OUT_F32, 2, 2),
    (264, 960, 5, 81, 77, capi.OUT_I8, 0, 2),
    (256, 1280, 10, 27, 31, capi.OUT_I8, 1, 2),   # from the kernel that reads the blob once
    (520, 264, 1, 13, 13, capi.OUT_I8, 0, 1),    # few values: one launch
])
def test_a_pointwise_layer_on_many_fp32_values(hip, C, K, n, h, w, kind, act, made):
    """A quantize pass and the launch with its operands in registers, where those are faster and there is room for the int8 blob: the bits of the
    single launch, which a caller without a workspace still gets."""
    rng = np.random.default_rng(C + K)
    conv = hip.conv(wq=rng.integers(-127, 128, (K, C, 1, 1)).astype(np.int8), scale_in=host_scale_in(np.full(K, 60.0, np.float32), 20.0),
                    bias=rng.normal(0, 1, K).astype(np.float32), in_scale=20.0, act=act, act_p0=0.1, out_kind=kind,
                    out_scale=[0.07] if kind == capi.OUT_I8 else None)
    x = hip.to_device((rng.integers(-260, 260, n * C * h * w) / np.float32(40)).astype(np.float32))  # ties and saturated values among them
    out_layout = capi.I8_P8 if kind == capi.OUT_I8 else capi.F32_P4
    got, count = _allocations(hip.torch, lambda: conv.forward(x, capi.F32_P8, n, h, w))
    assert count == made
    one = hip.torch.empty_like(got)
    assert hip.lib.otter_hip_conv_forward(conv.h, hip.ptr(x), capi.F32_P8, n, h, w, hip.ptr(one), out_layout, None, 0, hip.stream()) == 0
    assert hip.torch.equal(got, one)
    if x.numel() <= 32 << 20:
        assert hip.torch.equal(got, conv.forward_static(x, capi.F32_P8, n, h, w))  # (one launch: the array of all calls is not this layer's to write)
    conv.set_tile(-6, 0)
    assert hip.torch.equal(got, conv.forward(x, capi.F32_P8, n, h, w))
    conv.close()


def _pointwise_on_many_values(hip):
    """(layer, blob, batch, height, width, result) of a layer that is two launches where there is room for a workspace"""
    C, K, n, h, w = 520, 264, 24, 37, 53  # (a workspace of 24 MB: more than the allocator keeps beside what is in use)
    rng = np.random.default_rng(3)
    conv = hip.conv(wq=rng.integers(-127, 128, (K, C, 1, 1)).astype(np.int8), scale_in=host_scale_in(np.full(K, 60.0, np.float32), 20.0),
                    bias=rng.normal(0, 1, K).astype(np.float32), in_scale=20.0, act=3, out_kind=capi.OUT_I8, out_scale=[0.07])
    x = hip.to_device(rng.normal(0, 2, n * C * h * w).astype(np.float32))
    return conv, x, n, h, w, hip.empty(n * K * h * w, np.int8)


def test_an_error_of_the_workspace_allocation_is_the_calls(hip):
    """A workspace that such a layer could do without: an error that is not the lack of memory is raised, and none stays behind the call."""
    from torch.utils._python_dispatch import TorchDispatchMode

    conv, x, n, h, w, out = _pointwise_on_many_values(hip)

    class Refusing(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if "empty" in str(func):
                raise KeyError("no new tensors here")
            return func(*args, **(kwargs or {}))

    with Refusing(), pytest.raises(RuntimeError, match="no new tensors here"):
        conv.forward(x, capi.F32_P8, n, h, w, out=out)
    conv.forward(x, capi.F32_P8, n, h, w, out=out)
    conv.close()


@pytest.mark.parametrize("mode", [False, True])
def test_without_memory_for_a_workspace_it_is_one_launch(hip, mode):
    """Where there is no memory for a workspace that the layer can do without, the call does without it, also where a dispatch mode reports that."""
    import contextlib

    from torch.utils._python_dispatch import TorchDispatchMode

    torch = hip.torch
    conv, x, n, h, w, out = _pointwise_on_many_values(hip)
    want = conv.forward(x, capi.F32_P8, n, h, w)
    refused = []

    class Full(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            if "empty" in str(func):
                refused.append(func)
                raise torch.OutOfMemoryError("no memory")
            return func(*args, **(kwargs or {}))

    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_stats()["num_ooms"]
    try:
        if not mode:
            torch.cuda.set_per_process_memory_fraction(1e-9)  # (what is allocated stays; nothing more is given)
        with Full() if mode else contextlib.nullcontext():
            conv.forward(x, capi.F32_P8, n, h, w, out=out)
        assert len(refused) == mode and torch.cuda.memory_stats()["num_ooms"] - before == (not mode)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(out, want)
    conv.close()
