"""What the compiler is told and what it makes of the device code, on the CPU.

The compiler puts no wait states around an instruction inside an asm statement.
On gfx9 a vector memory instruction may read an SGPR that a vector instruction
(v_readlane, v_readfirstlane, a compare) wrote only five wait states later;
sooner it can see the old value, i.e. an address of two halves that do not
belong together. A base pointer reaches such an asm straight from v_readlane
whenever the register allocator parks SGPRs in lanes of a vector register, so
the source alone does not show it: the test compiles the unit as the build
does and reads the assembly.

Every attention kernel that a call can launch keeps the waves a SIMD it is
laid out for and uses no scratch memory, by the compiler's own account of it.

A forward call may write its output over Q, so the attention kernels that read
the 16-bit queries promise no aliasing for neither of the two pointers."""
from __future__ import annotations

import functools
import re
import subprocess

import pytest

import build as hip_build  # sota-papers-lab_amd/build.py

WAIT_STATES = 5  # VALU writes an SGPR, a VMEM instruction reads it


def _sgprs(text: str) -> set:
    out = {int(x) for x in re.findall(r"\bs(\d+)\b", text)}
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        out |= set(range(int(a), int(b) + 1))
    if "vcc" in text:
        out |= {"vcc"}
    return out


def sgpr_hazards(asm: str, need: int = WAIT_STATES) -> list:
    """(line, text) of every VMEM instruction that reads an SGPR fewer than
    `need` wait states after a VALU instruction wrote it, along straight-line
    code (a taken branch costs more than five)."""
    age, found = {}, []  # SGPR -> wait states since a VALU wrote it
    for n, line in enumerate(asm.splitlines(), 1):
        t = line.split(";")[0].strip()
        if not t or t.startswith(".") or t.startswith("//"):
            continue
        if t.endswith(":"):
            if not t.startswith(".L"):
                age = {}  # another function
            continue
        op, _, args = t.partition(" ")
        if re.match(r"(global|buffer|flat|scratch)_", op):
            if any(age.get(r, need) < need for r in _sgprs(args)):
                found.append((n, t))
        step = int(args, 0) + 1 if op == "s_nop" else 1
        age = {r: a + step for r, a in age.items() if a + step < need}
        dst = args.split(",")[0]
        written = _sgprs(dst)
        if op.startswith("v_"):
            # (carry-out and compare results name their SGPR second or first)
            if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[iu]64", op):
                written |= _sgprs(args.split(",")[1])
            age.update({r: 0 for r in written})
        else:
            for r in written:
                age.pop(r, None)  # a scalar write: interlocked
    return found


@functools.lru_cache(maxsize=None)
def assembly(unit: str, *flags: str) -> str:
    src, obj, extra = next(u for u in hip_build.UNITS if u[1] == unit)
    cmd = [hip_build.HIPCC, *hip_build.COMMON, *extra, "-x", "hip", "--cuda-device-only", "-S", *flags,
           str(hip_build.CSRC / src), "-o", "-"]
    return subprocess.run(cmd, check=True, capture_output=True, text=True, timeout=300).stdout


def test_the_scan_sees_a_short_wait():
    short = "f:\n v_readlane_b32 s3, v1, 2\n s_mov_b32 m0, s9\n s_nop 0\n global_load_lds_dwordx4 v1, s[2:3]\n"
    assert [n for n, _ in sgpr_hazards(short)] == [5]
    assert not sgpr_hazards(short.replace("s_nop 0", "s_nop 3"))
    assert not sgpr_hazards(short.replace("s_nop 0", "s_mov_b64 s[2:3], s[4:5]"))


UNITS_WITH_ASM = ["sage_attn_keys.hip.o"]


def test_only_these_units_load_in_inline_assembly():
    """Vector memory instructions inside asm statements: the shared helper and
    the keys-split kernels alone."""
    hits = {p.name for p in hip_build.CSRC.iterdir()
            if re.search(r'"(global|buffer|flat|scratch)_(load|store|atomic)', p.read_text())}
    assert hits == {"sage_attn_keys.hip", "sage_attn_device.hpp"}, hits


@pytest.mark.parametrize("unit", UNITS_WITH_ASM)
def test_vector_memory_waits_for_its_base(unit):
    asm = assembly(unit)
    assert "global_load_lds_dwordx4" in asm
    found = sgpr_hazards(asm)
    assert not found, f"{unit}: SGPR read too soon after a vector write: {found[:8]}"


@pytest.mark.parametrize("unit", UNITS_WITH_ASM)
def test_m0_belongs_to_the_asm_statements(unit):
    """The copies write M0 (their LDS base) without the compiler's knowledge:
    nothing it generates in the unit may hold a value there."""
    inside, other = False, []
    for n, line in enumerate(assembly(unit).splitlines(), 1):
        if "ASMSTART" in line or "ASMEND" in line:
            inside = "ASMSTART" in line
        elif not inside and re.search(r"\bm0\b", line.split(";")[0]):
            other.append((n, line.strip()))
    assert not other, f"{unit}: M0 used outside the asm statements: {other[:8]}"


@pytest.mark.parametrize("unit", ["sage_attention.hip.o", "sage_attention_merged.hip.o"])
def test_queries_and_output_may_alias(unit):
    """sage_attn<D, CAUSAL, MERGE, QF = true>(q, ..., out, geometry): the host
    launches it with out = q (q_readable_beside)."""
    ir = assembly(unit, "-emit-llvm", "-Xclang", "-disable-llvm-passes")
    seen = 0
    for args in re.findall(r"define [^@\n]*@_ZN4sage9sage_attnILi\d+ELb[01]ELb[01]ELb1EE\w*\(([^\n]*?)\) #", ir):
        ptrs = [a for a in args.split(", ") if "ptr" in a and "byref" not in a]
        assert len(ptrs) == 9, args
        for which in (0, 8):
            assert "noalias" not in ptrs[which], (which, ptrs[which])
        assert all("noalias" in p for p in ptrs[3:8])  # codes, scales and statistics: read only
        seen += 1
    assert seen == (2 if "merged" in unit else 4)


# VGPRs of the waves a SIMD each family is laid out for (512 a lane, in blocks
# of 8): 128 for four, 168 for three, 256 for two. Template arguments after the
# head dim: CAUSAL, MERGE, QF; CAUSAL, MERGE, shares, whole tiles beside them;
# CAUSAL.
WAVES = {
    r"9sage_attnILi64E": 128,
    r"9sage_attnILi128ELb[01]ELb0E": 168,
    r"9sage_attnILi128ELb0ELb1E": 256,
    r"14sage_attn_keysILi64ELb[01]ELb0E": 128,
    r"14sage_attn_keysILi64ELb0ELb1E": 168,
    r"14sage_attn_keysILi128ELb[01]ELb[01]ELi[24]ELb0E": 256,
    r"14sage_attn_keysILi128ELb0ELb0ELi4ELb1E": 168,
    r"15sage_attn_splitILi(64|128)E": 128,
}
KERNELS = {"sage_attention.hip.o": 12, "sage_attention_merged.hip.o": 4, "sage_attn_keys.hip.o": 10}


@pytest.mark.parametrize("unit", sorted(KERNELS))
def test_attention_kernels_fit(unit):
    meta = assembly(unit).split(".amdgpu_metadata")[1]
    kernels = re.split(r"\n  - ", meta)
    seen = 0
    for k in kernels:
        name = re.search(r"\.name:\s+(\S*sage_attn\S*)", k)
        if not name:
            continue
        get = lambda f: int(re.search(rf"\.{f}:\s+(\d+)", k).group(1))  # noqa: E731
        limit = [v for pat, v in WAVES.items() if re.search(pat, name.group(1))]
        assert len(limit) == 1, name.group(1)
        assert get("private_segment_fixed_size") == 0 and get("vgpr_spill_count") == 0, name.group(1)
        assert get("vgpr_count") <= limit[0], (name.group(1), get("vgpr_count"))
        seen += 1
    assert seen == KERNELS[unit]
