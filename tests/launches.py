"""The kernels that a call launches, by name."""
import pytest


def kernels(call):
    """Names of the device kernels that `call()` ran, in launch order."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA], acc_events=True) as prof:
        call()
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if "gfx::" in e.name]
    if not names:
        pytest.skip("the profiler reports no kernels here")
    return names
