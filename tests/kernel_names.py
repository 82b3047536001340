"""Names of the library's device kernels that a call launches, for tests of a dispatch
that no entry point names."""
from __future__ import annotations

import torch


def kernels(fn) -> list[str]:
    from torch.profiler import ProfilerActivity, profile

    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    return [e.name for e in prof.events() if "tvk::" in e.name]   # (host calls and torch's own kernels left out)
