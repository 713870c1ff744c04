"""The library's kernels that a call launches, by name (test helper)."""
import re
import warnings

import torch
from torch.profiler import ProfilerActivity, profile


def kernels(call):
    """(what call() returns, names of the library's kernels in the order of their launches, e.g. "gemm_split_kernel<8, 16, 32, 1, 0, 1>").
    No names where the profiler records nothing (another one holds the device): see expect."""
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        with profile(activities=[ProfilerActivity.CUDA]) as p:
            result = call()
            torch.cuda.synchronize()
    events = [e for e in p.events() if "qa::" in e.name and e.device_type == torch.autograd.DeviceType.CUDA]
    return result, [_plain(e.name) for e in sorted(events, key=lambda e: e.time_range.start)]


def _plain(name):
    name = re.sub(r"^void ", "", name).replace("(anonymous namespace)::", "")
    name = re.sub(r"\((?:qa::)?(?:\w+::)*\w+\)(?=\d)", "", name)              # (qa::split::ConvKind)1 -> 1
    return re.sub(r"(\w+::)+", "", re.match(r"[^(]*", name).group(0))


def expect(names, *starts):
    """The calls that a test is about were made of these kernels (prefixes of their names)."""
    if not names:
        warnings.warn("no kernel was recorded: the choice of the kernels is not checked")
        return
    for start in starts:
        assert any(n.startswith(start) for n in names), (start, names)
