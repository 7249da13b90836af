"""Which device work a call enqueues, by torch's profiler: for launch variants
whose results are the same by design."""


def device_events(f):
    """Names of the kernels and memory copies that f() runs on the GPU."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
        f()
        torch.cuda.synchronize()
    return [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA]
