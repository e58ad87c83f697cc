"""What the kernels' gfx950 assembly must and must not hold (CPU only: compiled
with the library's own flags). First the wait states that the hardware does not
check: a vector-memory instruction
may read a scalar register only five wait states or more after a vector ALU
instruction wrote it (AMD's CDNA instruction set guides, manually inserted
wait states). The compiler keeps that distance for its own instructions but
does not look into inline assembly, where the prefill issues its LDS copies."""
import functools
import re
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

from runtherder_amd import build as B

WAIT_STATES = 5
VMEM = re.compile(r"(global|buffer|scratch|flat)_")
ASM_SOURCES = [s for s in B.KERNEL_SOURCES
               if s.endswith(".hip") and "asm volatile" in (B.CSRC / s).read_text()]


def scalar_regs(operand):
    """Numbers of the scalar registers an operand names: s5, s[4:5], vcc is 106/107."""
    operand = operand.strip()
    if m := re.fullmatch(r"s(\d+)", operand):
        return {int(m[1])}
    if m := re.fullmatch(r"s\[(\d+):(\d+)\]", operand):
        return set(range(int(m[1]), int(m[2]) + 1))
    return {106, 107} if operand.startswith("vcc") else set()


def instructions(asm):
    """(mnemonic, operands) per instruction, in order; function bounds as (None, [])."""
    out = []
    for line in asm.splitlines():
        line = line.split(";")[0].strip()
        if re.match(r"[_A-Za-z]\S*:", line) and not line.startswith(".L"):
            out.append((None, []))
        elif line and not line.startswith(".") and not line.endswith(":"):
            name, _, rest = line.partition(" ")
            out.append((name, [o.strip() for o in rest.split(",")]))
    return out


def short_distances(asm):
    """Vector-memory instructions that read a scalar register too soon after a
    vector ALU write of it, along the instruction order."""
    seq, bad, seen = instructions(asm), [], 0
    for i, (name, ops) in enumerate(seq):
        if name is None or not VMEM.match(name):
            continue
        reads = set().union(*(scalar_regs(o.split(" ")[0]) for o in ops))
        if not reads:
            continue
        seen += 1
        states, j = 0, i - 1
        while j >= 0 and states < WAIT_STATES and seq[j][0] is not None and reads:
            wname, wops = seq[j]
            writes = scalar_regs(wops[0]) if wops else set()
            if wname.startswith("v_") and writes & reads:
                bad.append(f"{wname} {', '.join(wops)} -> {name} {', '.join(ops)}: {states}")
                break
            reads = reads - writes   # a later scalar write: the hardware orders that itself
            states += int(wops[0]) + 1 if wname == "s_nop" else 1
            j -= 1
    return bad, seen


def test_the_check_sees_a_short_distance():
    head = "k:\n v_readfirstlane_b32 s4, v2\n v_readfirstlane_b32 s5, v3\n s_mov_b32 m0, s9\n"
    load = " global_load_lds_dwordx4 v1, s[4:5]\n"
    assert len(short_distances(head + " s_nop 0\n" + load)[0]) == 1
    assert not short_distances(head + " s_nop 3\n" + load)[0]
    assert not short_distances(head + " s_mov_b64 s[4:5], s[4:5]\n" + load)[0]
    assert short_distances(head + " s_nop 3\n" + load)[1] == 1


@functools.lru_cache(maxsize=None)
def assembly(src):
    flags = [f for f in B.DEVICE_FLAGS if f != "-fPIC"]
    with tempfile.TemporaryDirectory() as d:
        out = Path(d) / "k.s"
        res = subprocess.run([B.HIPCC, *flags, "-x", "hip", "--cuda-device-only", "-S",
                              str(B.CSRC / src), "-o", str(out)], capture_output=True, text=True)
        assert res.returncode == 0, res.stderr[-2000:]
        return out.read_text()


needs_hipcc = pytest.mark.skipif(shutil.which(B.HIPCC) is None and not Path(B.HIPCC).exists(),
                                 reason="hipcc not available")


@needs_hipcc
@pytest.mark.parametrize("src", ASM_SOURCES)
def test_scalar_bases_of_memory_instructions_have_settled(src):
    bad, seen = short_distances(assembly(src))
    assert seen > 50, f"only {seen} memory instructions with a scalar base parsed"
    assert not bad, f"{len(bad)} of {seen}: " + "; ".join(bad[:4])


@needs_hipcc
def test_prefill_tile_loop_waits_for_no_scalar_load():
    """The prefill's tile loop (it holds the third barrier of each kernel) has no
    scalar load, whose round trip every tile would wait for, and takes values out
    of vector registers only for a paged cache's two block-table entries."""
    text, seen = assembly("flash_prefill.hip"), 0
    for m in re.finditer(r"^(_Z\w*flash_prefill_kernelILi\dELb(\d)\w*):.*?^\.Lfunc_end", text,
                         re.M | re.S):
        code = [line.split(";")[0].strip() for line in m[0].splitlines()]
        at = [i for i, line in enumerate(code) if line == "s_barrier"][2]
        # From the loop's head (the target of the first branch back past the barrier).
        label = {line[:-1]: i for i, line in enumerate(code) if re.match(r"\.LBB\w+:", line)}
        end, head = next((i, label[t[1]]) for i, line in enumerate(code[at:], at)
                         if (t := re.match(r"s_c?branch\w* (\.LBB\w+)", line)) and label[t[1]] < at)
        loop = code[head:end]
        assert sum("mfma" in line for line in loop) == 24, m[1]
        assert not [line for line in loop if line.startswith("s_load")], m[1]
        taken = sum(line.startswith("v_readfirstlane") for line in loop)
        assert taken == (2 if m[2] == "1" else 0), (m[1], taken)
        seen += 1
    assert seen == 6
