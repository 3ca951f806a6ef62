"""The native call path's allocations: what torch offers to see or to change an allocation sees these too."""
import numpy as np
import pytest

from tensor_amd import capi

pytestmark = pytest.mark.gpu


def test_allocations_are_visible_to_modes_and_profilers(hip):
    from torch.utils._python_dispatch import TorchDispatchMode
    torch = hip.torch
    rng = np.random.default_rng(0)
    conv = hip.conv(wq=rng.integers(-127, 128, (16, 16, 3, 3)).astype(np.int8), scale_in=np.full(16, 1e-3, np.float32), pad=(1, 1),
                    out_kind=capi.OUT_F32)
    x = hip.to_device(rng.integers(-127, 128, 16 * 81).astype(np.int8))
    want = conv.forward(x, capi.I8_P8, 1, 9, 9)
    calls = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            calls.append(str(func))
            return func(*args, **(kwargs or {}))

    with Watch():
        got = conv.forward(x, capi.I8_P8, 1, 9, 9)
    assert any("empty" in c for c in calls) and torch.equal(got, want)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        got = conv.forward(x, capi.I8_P8, 1, 9, 9)
    assert any("empty" in e.name for e in prof.events()) and torch.equal(got, want)
    before = torch.are_deterministic_algorithms_enabled()
    torch.use_deterministic_algorithms(True)
    try:
        assert torch.equal(conv.forward(x, capi.I8_P8, 1, 9, 9), want)
    finally:
        torch.use_deterministic_algorithms(before)
    with torch.inference_mode():
        got = conv.forward(x, capi.I8_P8, 1, 9, 9)
        assert got.is_inference() and torch.equal(got, want)
    conv.close()
