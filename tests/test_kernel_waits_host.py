"""Host-side check of the device code of the MX GEMM kernels: the K loop of a persistent kernel
must not contain a vector-memory wait that the compiler added on its own.

The kernels wait for their direct-to-LDS copies with hand-written ``s_waitcnt vmcnt(N)``
instructions inside ``asm`` statements, which leave copies of later slabs in flight. The
compiler's own wait-count bookkeeping does not see those; if it believes that a vector load of
the epilogue may still be outstanding when the K loop of the next tile begins (a load and its use
in two separately guarded blocks are enough), it puts an ``s_waitcnt vmcnt(0)`` in front of the
first instruction of the loop that overwrites the load's register -- and every slab then begins by
waiting for all copies in flight (dense MXFP8 16384^3: 3.2 -> 3.7 ms). The test compiles the
translation units to assembly (no GPU needed) and looks at the MFMA loops of their kernels.

The same assembly goes through what the build looks for in it (check_asm.py)."""

import re
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "primus-turbo_amd"))
import check_asm  # noqa: E402


def _innermost_mfma_loops(body):
    labels = {m.group(1): i for i, l in enumerate(body) if (m := re.match(r"^(\.LBB\d+_\d+):", l))}
    loops = []
    for i, l in enumerate(body):
        m = re.match(r"\s+s_cbranch_\w+ (\.LBB\d+_\d+)", l)
        if m and labels.get(m.group(1), i) < i:
            loops.append((labels[m.group(1)], i))
    with_mfma = [(s, e) for s, e in loops if sum("v_mfma" in x for x in body[s:e]) >= 16]
    return [(s, e) for s, e in with_mfma if not any(s < s2 and e2 < e for s2, e2 in with_mfma)]


def _compiler_vmcnt_waits(seg):
    """``s_waitcnt`` instructions with a vmcnt field outside the kernel's own asm statements."""
    out, in_asm = [], False
    for x in seg:
        if "#ASMSTART" in x:
            in_asm = True
        elif "#ASMEND" in x:
            in_asm = False
        elif not in_asm and "s_waitcnt" in x and "vmcnt" in x:
            out.append(x.strip())
    return out


def _copy(nop=0, descriptor="s[0:3]"):
    return ["\t;;#ASMSTART", "\ts_add_u32 m0, s4, 16", f"\ts_nop {nop}", f"\tbuffer_load_dword v1, {descriptor}, 0 offen lds", "\t;;#ASMEND"]


@pytest.mark.parametrize("write,caught", [("v_readlane_b32 s3, v2, 0", True), ("v_readlane_b32 s4, v2, 0", False),
                                          ("v_readfirstlane_b32 s0, v2", True), ("v_cmp_lt_u32_e64 s[2:3], v1, v2", True),
                                          ("v_add_co_u32_e64 v1, s[0:1], v1, v2", True), ("v_add_u32_e32 v1, s0, v2", False),
                                          ("s_mov_b32 s0, s7", False)])
def test_check_sees_a_short_wait(write, caught):
    three = ["\ts_nop 1", "\ts_mov_b32 s9, s8"]
    fault = ["less than 5 wait states from a VALU write of the descriptor: buffer_load_dword v1, s[0:3], 0 offen lds"]
    found = (1, fault if caught else [])
    assert check_asm.faults_of_copies(["\t" + write] + _copy()) == found
    assert check_asm.faults_of_copies(["\t" + write] + three[:1] + _copy()) == found  # (four states)
    assert check_asm.faults_of_copies(["\t" + write] + three + _copy()) == (1, [])  # (five)
    # on the way of a jump, and behind one that does not come here
    loop = [".LBB0_1:"] + _copy() + ["\ts_nop 7", "\t" + write, "\ts_cbranch_scc0 .LBB0_1"]
    assert check_asm.faults_of_copies(loop) == found
    assert check_asm.faults_of_copies(["\t" + write, "\ts_branch .LBB0_2", ".LBB0_1:"] + _copy()) == (1, [])


def test_check_sees_another_use_of_m0():
    assert check_asm.faults_of_copies(_copy() + ["\ts_mov_b32 m0, s7 ; m0"]) == (1, ["M0 is used besides the copies: s_mov_b32 m0, s7"])
    assert check_asm.faults_of_copies(["\ts_mov_b32 m0, s7", "\tbuffer_load_dword v1, s[0:3], 0 offen lds"]) == (0, [])


def test_scanner_sees_a_compiler_wait():
    body = [".LBB0_1:"] + ["\tv_mfma_f32 a, b, c"] * 16 + ["\t;;#ASMSTART", "\ts_waitcnt vmcnt(3)", "\t;;#ASMEND",
                                                          "\ts_waitcnt vmcnt(0)", "\ts_cbranch_scc0 .LBB0_1"]
    (s, e), = _innermost_mfma_loops(body)
    assert _compiler_vmcnt_waits(body[s:e]) == ["s_waitcnt vmcnt(0)"]


# translation unit -> which of its kernels are looked at: the dense MX kernels (gemm_mx8_kernel and
# gemm_fp8_nt_kernel<TM, TN, 2 = MX, ...>), the block-scaled eight-wavefront kernel of the
# headline workload (the four-wavefront block kernels of that unit load their scales into
# registers inside the loop and wait for them legitimately), its grouped form, the grouped vector-scale kernels
# and those that transpose an operand as they read it; and how many MFMA loops they have at least
UNITS = {
    "gemm_mx.hip": (lambda n: "gemm_mx8_kernel" in n or re.search(r"gemm_fp8_nt_kernelILi\dELi\dELi2E", n), 8),
    "gemm_fp8_block.hip": (lambda n: "gemm_fp8_block8_kernel" in n, 4),
    # vector scales (tensorwise / rowwise), row groups and variable K: the epilogue loads its scales
    "gemm_fp8_grouped_vec.hip": (lambda n: re.search(r"gemm_fp8_nt_kernelILi\dELi\dELi0E", n), 8),
    "gemm_fp8_grouped.hip": (lambda n: "gemm_fp8_block8_kernel" in n, 8),
    "gemm_fp8_kn.hip": (lambda n: "gemm_fp8_nt_kernel" in n, 8),
    "gemm_mx_grouped_kn.hip": (lambda n: "gemm_fp8_nt_kernel" in n, 10),
}
# those of them with copies in asm statements, and in how many kernels
COPIES = {"gemm_fp8_block.hip": 4, "gemm_fp8_grouped.hip": 4, "gemm_fp8_kn.hip": 8, "gemm_mx_grouped_kn.hip": 10}


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    """Device assembly of the units, compiled side by side (about three minutes of hipcc)."""
    from concurrent.futures import ThreadPoolExecutor

    import build_native

    try:
        hipcc = build_native.hipcc_path()
    except RuntimeError:
        pytest.skip("hipcc not found")
    out = tmp_path_factory.mktemp("asm")
    flags = [f for f in build_native.HIPCC_FLAGS if f != "-fPIC"]

    def one(unit):
        src = build_native.CSRC / unit
        asm = out / (src.stem + ".s")
        cmd = [hipcc, *flags, *build_native._extra_flags(src), "-S", "--cuda-device-only", "-o", str(asm), str(src)]
        res = subprocess.run(cmd, capture_output=True, text=True)
        assert res.returncode == 0, res.stderr[-2000:]
        return unit, asm.read_text().split("\n")

    with ThreadPoolExecutor(max_workers=len(UNITS)) as ex:
        return dict(ex.map(one, UNITS))


@pytest.mark.parametrize("unit", sorted(UNITS))
def test_mfma_loops_have_no_compiler_inserted_vmcnt_wait(assembly, unit):
    lines = assembly[unit]
    wanted, least = UNITS[unit]
    seen, bad = 0, []
    for name, a, b in check_asm.functions(lines):
        if not wanted(name):
            continue
        body = lines[a:b]
        for s, e in _innermost_mfma_loops(body):
            seen += 1
            waits = _compiler_vmcnt_waits(body[s:e])
            if waits:
                bad.append((name, waits))
    assert seen >= least, f"only {seen} MFMA loops found: the scanner no longer matches the compiler's output"
    assert not bad, bad


@pytest.mark.parametrize("unit", sorted(UNITS))
def test_copies_are_checked(assembly, unit):
    lines, kernels = assembly[unit], 0
    for name, a, b in check_asm.functions(lines):
        copies, faults = check_asm.faults_of_copies(lines[a:b])
        kernels += copies > 0
        assert not faults, (name, faults[:5])
    assert kernels == COPIES.get(unit, 0)
