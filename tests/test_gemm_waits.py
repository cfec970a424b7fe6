"""Waits that the fragment GEMM's inline assembly owes the hardware, read from
the disassembly of the built library (no GPU needed): the compiler's own wait
insertion does not look into inline assembly."""
import os
import re
import shutil
import struct
import subprocess

import pytest

import cbq_native as nat

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(lib):
    """The gfx950 code objects bundled in a shared library."""
    data, at = open(lib, "rb").read(), 0
    while (at := data.find(MAGIC, at)) >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + idlen]:
                yield data[at + off:at + off + size]
            p += 24 + idlen
        at += len(MAGIC)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{symbol: [instruction, ...]} of every frag_gemm_kernel."""
    if not os.path.exists(nat.SO_PATH) or not os.path.exists(OBJDUMP):
        pytest.skip("needs the built library and llvm-objdump")
    out = {}
    for i, co in enumerate(_code_objects(nat.SO_PATH)):
        if b"frag_gemm_kernel" not in co:
            continue
        f = tmp_path_factory.mktemp("co") / f"{i}.co"
        f.write_bytes(co)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(f)], check=True,
                              capture_output=True, text=True).stdout
        name = None
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(.*)>:", line)
            if m:
                name = m.group(1)
            elif name and "frag_gemm_kernel" in name and line.startswith("\t"):
                out.setdefault(name, []).append(line.split("//")[0].strip())
        shutil.rmtree(f.parent)
    assert out, "no frag_gemm_kernel in the library"
    return out


def _sgprs(text):
    regs = set()
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        regs |= set(range(int(a), int(b) + 1))
    return regs | {int(r) for r in re.findall(r"\bs(\d+)\b", text)}


def test_copy_addresses_wait_for_valu_writes(kernels):
    """A VMEM instruction may read a scalar register five wait states after a
    VALU instruction wrote it, no sooner (CDNA3 ISA guide, manually inserted
    wait states); one instruction is one state, s_nop N is N + 1."""
    copies, early = 0, []
    for name, ins in kernels.items():
        for i, line in enumerate(ins):
            if not line.startswith("global_load_lds"):
                continue
            copies += 1
            need, states = _sgprs(line.split(None, 1)[1]), 0
            for prev in reversed(ins[max(0, i - 5):i]):
                if states >= 5:
                    break
                op, _, args = prev.partition(" ")
                if op.startswith("v_") and _sgprs(args.split(",")[0]) & need:
                    early.append((name, prev, line))
                states += int(args, 0) + 1 if op == "s_nop" else 1
    assert copies > 100
    assert not early, f"{len(early)} of {copies}: {early[0]}"


def test_barriers_bound_the_lds_reads(kernels):
    """The barrier before a stage's LDS is written again waits for the reads
    of that stage: each carries a bound on the LDS reads in flight.  At most
    the 12 of a stage's first product (8 + 4 fragments) may be newer."""
    barriers = 0
    for name, ins in kernels.items():
        for i, line in enumerate(ins):
            if line != "s_barrier":
                continue
            barriers += 1
            m = re.search(r"lgkmcnt\((\d+)\)", ins[i - 1])
            assert ins[i - 1].startswith("s_waitcnt") and m and int(m.group(1)) <= 12, \
                (name, ins[i - 1])
    assert barriers > 40
