"""Which device work a call enqueues, by torch's profiler: for launch variants
whose results are the same by design."""
import time


def device_events(f, expected=()):
    """Names of the kernels and memory copies that f() runs on the GPU.  The
    profiler drops events that its clocks place outside the recorded interval,
    hence the margins, and f() is repeated until every text of `expected` is
    part of some name, at most 5 times."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    names = []
    for _ in range(5):
        torch.cuda.synchronize()
        with profile(activities=[ProfilerActivity.CPU, ProfilerActivity.CUDA]) as prof:
            time.sleep(0.02)
            f()
            torch.cuda.synchronize()
            time.sleep(0.02)
        names += [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA]
        if all(any(x in n for n in names) for x in expected):
            break
    return names
