"""What the built library's attention kernels take of a wavefront's private memory.  A register read back from there waits for all copies in
flight (loads complete in order), so they spill none in their loops: a few have one or two that are stored before the loop and read after it, and
a change that brings more is to be looked at."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import _capi

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _readelf():
    for path in (shutil.which("llvm-readelf"), "/opt/rocm/llvm/bin/llvm-readelf"):
        if path and os.path.exists(path):
            return path
    return None


def _code_objects(data):
    """The gfx950 code objects of the library's bundles (one for each source): a bundle is the magic, the number of entries and for
    each its offset in the bundle, its size and its target."""
    at = data.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, p)
            target = data[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" in target and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


def test_registers_spilled(tmp_path):
    tool = _readelf()
    if tool is None:
        pytest.skip("no llvm-readelf")
    kernels = {}
    for i, obj in enumerate(_code_objects(open(_capi.LIB, "rb").read())):
        path = tmp_path / f"{i}.o"
        path.write_bytes(obj)
        notes = subprocess.run([tool, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for part in notes.split("  - .agpr_count:")[1:]:                      # one for each kernel
            name = re.search(r"^ +\.name: +(\S+)", part, re.M)[1]
            kernels[name] = tuple(int(re.search(rf"\.{key}: +(\d+)", part)[1]) for key in ("vgpr_spill_count", "private_segment_fixed_size"))
    attention = {n: v for n, v in kernels.items() if "attn_" in n}
    assert len(attention) > 100
    assert {n: v for n, v in attention.items() if v[0] > 2 or v[1] > 12} == {}
