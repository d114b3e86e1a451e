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


def _forward_kernels(tmp_path, named):
    """{demangled template arguments: instructions} of the library's forward kernels whose arguments `named` accepts."""
    objdump = os.path.join(os.path.dirname(_readelf() or ""), "llvm-objdump")
    if not os.path.exists(objdump) or shutil.which("c++filt") is None:
        pytest.skip("no llvm-objdump")
    found = {}
    for i, obj in enumerate(_code_objects(open(_capi.LIB, "rb").read())):
        if b"attn_fwd_kernel" not in obj:
            continue
        path = tmp_path / f"{i}.o"
        path.write_bytes(obj)
        symbols = re.findall(r"FUNC .* (\S*attn_fwd_kernel\S*)$", subprocess.run([_readelf(), "-sW", str(path)], capture_output=True, text=True, check=True).stdout, re.M)
        names = subprocess.run(["c++filt"] + symbols, capture_output=True, text=True, check=True).stdout.split("\n")
        wanted = {s: re.search(r"attn_fwd_kernel<(.*?)>", n)[1] for s, n in zip(symbols, names)}
        wanted = {s: n for s, n in wanted.items() if named(n.split(", "))}
        if wanted:
            text = subprocess.run([objdump, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + ",".join(wanted), str(path)], capture_output=True, text=True, check=True).stdout
            for part in text.split("\n\n"):
                head = re.search(r"<(\S+)>:$", part, re.M)
                if head and head[1] in wanted:
                    found[wanted[head[1]]] = [line.split("//")[0].strip() for line in part[head.end():].strip().split("\n")]
    return found


# BF16, POSTMUL, PACKED_ROWS, head dim, BYTEMASK, BYPRODUCTS, FETCH, SPLIT, WIDE_Q, HALVES
def test_forward_requests_its_queries_at_once(tmp_path):
    """A wavefront's q fragments come from LDS in one round trip, not in one for each: they are all requested before the first is waited for.
    (One after the other they cost a call of two tiles 0.08 us of 4.6, and 16 rows of head dim 128 0.13 of 5.5.)"""
    kernels = _forward_kernels(tmp_path, lambda n: n[:3] == ["false", "false", "true"] and n[5] == n[8] == "false")
    assert len(kernels) > 20
    for name, code in kernels.items():
        first = next(i for i, c in enumerate(code) if c.startswith("ds_read_b128"))
        wait = next(i for i, c in enumerate(code) if i > first and c.startswith("s_waitcnt") and "lgkmcnt" in c)
        reads = sum(c.startswith("ds_read_b128") for c in code[first:wait])
        assert reads >= 2 * int(name.split(", ")[3]) // 32, (name, reads)


def test_forward_asks_for_what_its_end_needs_late(tmp_path):
    """Arguments come from the host's memory, and no copy is requested before those asked for at the start are there: what only the end of the forward
    needs (the outputs) is asked for behind the first copies, and the grid's size, which lies behind all arguments, not at all.
    (All at the start cost a small call 0.15 to 0.25 us of 5.)"""
    source = tmp_path / "offsets.cpp"
    source.write_text('#include <stdio.h>\n#include <stddef.h>\n#include "sma_internal.h"\n'
                      'int main() { using A = sma::AttnArgs; printf("%zu %zu %zu", offsetof(A, out), offsetof(A, lse), sizeof(A)); }\n')
    csrc = os.path.join(os.path.dirname(_capi.LIB), "csrc")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include", "-I" + csrc, str(source), "-o", str(tmp_path / "offsets")], check=True)
    out, lse, size = map(int, subprocess.run([str(tmp_path / "offsets")], capture_output=True, text=True, check=True).stdout.split())
    kernels = _forward_kernels(tmp_path, lambda n: n[:3] == ["false", "false", "true"] and n[5] == n[8] == "false")
    assert len(kernels) > 20
    for name, code in kernels.items():
        copy = next(i for i, c in enumerate(code) if c.startswith("global_load_lds"))
        asked = set()
        for c in code[:copy]:
            m = re.match(r"s_load_dword(?:x(\d+))? s(?:\[\d+:\d+\]|\d+), s\[0:1\], (0x[0-9a-f]+)", c)
            if m:
                at = int(m[2], 16)
                asked |= set(range(at, at + 4 * int(m[1] or 1), 4))
        assert asked, name
        assert not asked & {lse, *range(out, out + 20, 4)}, name
        assert name.split(", ")[7] == "true" or max(asked) < size, name


def test_forward_requests_the_pieces_of_a_row_together(tmp_path):
    """At head dim 96 a row of K or V is copied in two pieces, 128 bytes and 64: those of K, then those of V, since a row's end and the next row's begin lie
    in the same lines.  (The ends after both cost 384 heads of 112 rows 0.25 us of 8.85.)"""
    kernels = _forward_kernels(tmp_path, lambda n: n[:4] == ["false", "false", "true", "96"] and n[7] == n[8] == "false")
    assert len(kernels) >= 6
    for name, code in kernels.items():
        bases = [re.search(r"(s\[\d+:\d+\])", c)[1] for c in code if c.startswith("global_load_lds_dwordx4")]
        # (six copies of q first; the boolean mask's, one or two a tile and of another base, are no part of this)
        q, rest = bases[:6], bases[6:]
        if name.split(", ")[4] == "false":
            assert len(rest) % 6 == 0, (name, rest)
            tiles = [rest[i:i + 6] for i in range(0, len(rest), 6)]
        else:
            copies = 6 + (1 if name.split(", ")[9] == "true" and name.split(", ")[5] == "false" else 2)
            assert len(rest) % copies == 0, (name, rest)
            tiles = [rest[i:i + 6] for i in range(0, len(rest), copies)]
        assert tiles and len(set(q)) == 1, name
        assert all(t[0] == t[1] == t[2] and t[3] == t[4] == t[5] for t in tiles), (name, tiles)


def test_lds_of_the_value_fragments(tmp_path):
    """dK/dV with V's fragments in LDS: a wavefront's area holds what it writes there, two fragments of 1 KiB for each step of 32 columns, at every head dim."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    source = tmp_path / "frag.hip"
    source.write_text('#include "attn_bwd.hip"\n'
                      "template <int HDIM> constexpr bool holds() { return sma::DkvCfg<HDIM, 4, true>::FRAG >= 2 * ((HDIM + 31) / 32) * 1024; }\n"
                      'static_assert(holds<32>() && holds<64>() && holds<80>() && holds<96>() && holds<128>(), "V fragments");\n')
    csrc = os.path.join(os.path.dirname(_capi.LIB), "csrc")
    include = os.path.join(os.path.dirname(os.path.dirname(_capi.LIB)), "include")
    subprocess.run([hipcc, "--offload-host-only", "-fsyntax-only", "-std=c++17", "-I" + include, "-I" + csrc, str(source)], check=True)
