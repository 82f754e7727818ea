"""Wait states behind the matrix instructions of the built library, along all paths.

The result of an FP64 16x16x4 matrix instruction may be read 18 wait states after it (FP32: 10)
and its register written again by the vector ALU after 11 (FP32: 10); an instruction is
one state, s_nop N is N + 1.  The compiler counts them, but was seen to count too few where
the use lies behind a taken branch.
"""
import os
import re
import struct
import subprocess

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hfem_amd", "libhfem_amd.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
READ, REWRITE = {"f64": 18, "f32": 10}, {"f64": 11, "f32": 10}
REG = re.compile(r"\b([va])(?:(\d+)|\[(\d+):(\d+)\])(?!\w)")
MEMORY = ("ds_", "global_", "buffer_", "flat_", "scratch_")
# instructions whose first operand is read
SOURCES_ONLY = ("ds_write", "s_", "v_cmp", "v_readlane", "v_readfirst", "ds_add", "ds_max", "global_atomic")


def code_objects(data):
    """The gfx950 code objects of the library's offload bundles."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        (count,), p = struct.unpack_from("<Q", data, at + 24), at + 32
        for _ in range(count):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length]:
                yield data[at + off:at + off + size]
            p += 24 + length
        at += 24


def regs(text):
    out = set()
    for kind, one, lo, hi in REG.findall(text):
        out.update((kind, i) for i in (range(int(lo), int(hi) + 1) if lo else [int(one)]))
    return out


def operands(name, ops):
    """Registers an instruction writes and those it reads (a matrix instruction's addend, which
    the hardware forwards, left out)."""
    first, _, rest = ops.partition(",")
    if "mfma" in name:
        a, b = rest.split(",")[:2]
        return regs(first), regs(a) | regs(b)
    if "store" in name or name.startswith(SOURCES_ONLY) or name.startswith("buffer_") and "lds" in ops:
        return set(), regs(ops)
    reads = regs(rest)
    if name.startswith(("v_fmac", "v_swap")) or "dpp" in name or "row_" in ops:
        reads |= regs(first)
    return regs(first), reads


def short_waits(listing):
    """(kernel, matrix instruction, use, states) of every use that comes too early."""
    bad = []
    for part in re.split(r"\n(?=[0-9a-f]+ <)", listing):
        head = re.match(r"[0-9a-f]+ <(\S+)>:", part)
        if not head or "mfma" not in part:
            continue
        code, at = [], {}
        for line in part.splitlines()[1:]:
            m = re.match(r"\s+(\w+)(.*?)\s*// ([0-9A-F]+):.*?(?:<\S+\+0x([0-9a-f]+)>)?$", line)
            if m:
                at[int(m[3], 16)] = len(code)
                code.append((m[1], m[2].strip(), m[4]))
        base = min(at)
        parsed = {}
        for start, (name, ops, _) in enumerate(code):
            if "mfma" not in name:
                continue
            kind = "f64" if "f64" in name else "f32"
            paths, seen = [(start + 1, 0, frozenset(operands(name, ops)[0]))], {}
            while paths:
                i, states, live = paths.pop()
                # (a place reached again later, with no more registers, adds nothing)
                if states >= READ[kind] or not live or i >= len(code) or \
                        i in seen and seen[i][0] <= states and live <= seen[i][1]:
                    continue
                seen[i] = states, live
                op, args, target = code[i]
                if op == "s_nop":
                    paths.append((i + 1, states + int(args, 0) + 1, live))
                    continue
                if op in ("s_endpgm", "s_setpc_b64"):
                    continue
                if op.startswith(("s_branch", "s_cbranch")):
                    paths.append((at[base + int(target or "0", 16)], states + 1, live))
                    if op != "s_branch":
                        paths.append((i + 1, states + 1, live))
                    continue
                if i not in parsed:
                    parsed[i] = operands(op, args)
                writes, reads = parsed[i]
                rewrite = not op.startswith(MEMORY) and "mfma" not in op and states < REWRITE[kind]
                if live & reads or rewrite and live & writes:
                    bad.append((head[1], f"{name} {ops}", f"{op} {args}", states))
                paths.append((i + 1, states + 1, live - writes))
    return bad


def test_planted():
    """A use behind a taken branch is found: 17 states behind the branch, 18 without it."""
    text = ("0000000000001000 <k>:\n\tv_mfma_f64_16x16x4_f64 v[0:7], v[8:9], v[10:11], v[0:7] // 000000001000: 00\n"
            "\ts_cbranch_execz 1 // 000000001008: 00 <k+0x10>\n" + "\ts_nop 0 // 00000000100C: 00\n"
            + "\ts_nop 15 // 000000001010: 00\n" + "\tds_write_b64 v20, v[2:3] // 000000001014: 00\n"
            + "\ts_endpgm // 000000001018: 00\n")
    assert [b[3] for b in short_waits(text)] == [17]
    assert not short_waits(text.replace("s_nop 0 ", "s_nop 1 ").replace("execz 1 // 000000001008: 00 <k+0x10>",
                                                                         "execz 0 // 000000001008: 00 <k+0xc>"))


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_library(tmp_path):
    if not os.path.exists(LIB):
        from hfem_amd import build
        build.build()
    kernels, bad = 0, []
    for i, obj in enumerate(code_objects(open(LIB, "rb").read())):
        path = tmp_path / f"{i}.co"
        path.write_bytes(obj)
        listing = subprocess.run([OBJDUMP, "-d", str(path)], capture_output=True, text=True, check=True).stdout
        kernels += listing.count("mfma") > 0
        bad += short_waits(listing)
    assert kernels >= 5
    assert not bad, f"{len(bad)} uses too early, the first: " + "; ".join(map(str, bad[:8]))
