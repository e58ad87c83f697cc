"""Wait states that the hardware does not check (CPU only: compiles the kernels
to gfx950 assembly with the library's own flags). A vector-memory instruction
may read a scalar register only five wait states or more after a vector ALU
instruction wrote it (AMD's CDNA instruction set guides, manually inserted
wait states). The compiler keeps that distance for its own instructions but
does not look into inline assembly, where the prefill issues its LDS copies."""
import re
import shutil
import subprocess
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


@pytest.mark.skipif(shutil.which(B.HIPCC) is None and not Path(B.HIPCC).exists(),
                    reason="hipcc not available")
@pytest.mark.parametrize("src", ASM_SOURCES)
def test_scalar_bases_of_memory_instructions_have_settled(src, tmp_path):
    out = tmp_path / "k.s"
    flags = [f for f in B.DEVICE_FLAGS if f != "-fPIC"]
    res = subprocess.run([B.HIPCC, *flags, "-x", "hip", "--cuda-device-only", "-S",
                          str(B.CSRC / src), "-o", str(out)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    bad, seen = short_distances(out.read_text())
    assert seen > 50, f"only {seen} memory instructions with a scalar base parsed"
    assert not bad, f"{len(bad)} of {seen}: " + "; ".join(bad[:4])
