"""Which kernels a call launches, for tests that are about one of them: a rule that sends their sizes elsewhere is then noticed."""
import json
import os
import re
import tempfile
import warnings

import torch


def launches(fn):
    """[(kernel, template arguments, work-groups)] of the library's kernels that fn() launches, in order."""
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
            fn()
            torch.cuda.synchronize()
    fd, path = tempfile.mkstemp(suffix=".json")
    os.close(fd)
    try:
        prof.export_chrome_trace(path)
        with open(path) as f:
            events = [e for e in json.load(f)["traceEvents"] if e.get("cat") == "kernel"]
    finally:
        os.remove(path)
    found = []
    for e in sorted(events, key=lambda e: e["ts"]):
        m = re.search(r"sma::\(anonymous namespace\)::(\w+?)(?:<([^>]*)>)?\(", e["name"])
        if m:
            found.append((m[1], tuple(t.strip() for t in (m[2] or "").split(",")), int(e["args"]["grid"][0])))
    return found


def places():
    """Work-groups of which a CU holds one: the places of a round."""
    return torch.cuda.get_device_properties(0).multi_processor_count
