"""Static check of the inline-assembly fragment reads in the 256 x 256 GEMM (CPU only).

The k-loop issues all of its fragment reads as inline assembly (``ds_read_b64_tr_b16`` of an
M/N-contiguous operand, ``ds_read_b128`` of a K-contiguous one), which the compiler does not
know to be LDS loads: it inserts no wait before their results are used. Their results become
usable only at the explicit ``s_waitcnt lgkmcnt(0)`` that follows them (``tie_wait``). Until
then no instruction may read or write a destination register of a pending read, and no branch
may leave with one pending. The GPU tests check the results; this test compiles the kernels
to gfx950 assembly with the library's build flags and checks that rule on every
instantiation, so that a compiler that moves or copies a fragment register ahead of its wait
fails here, before any GPU run. (The epilogues' own LDS reads go through the compiler, which
waits for them itself, with counted waits that this check does not model.)
"""
import re
import shutil
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
PACKAGE = ROOT / "warpstate-ai_amd"
sys.path.insert(0, str(PACKAGE))

import build_lib  # noqa: E402

HIPCC = shutil.which(build_lib.HIPCC) or (build_lib.HIPCC if Path(build_lib.HIPCC).exists() else None)
pytestmark = pytest.mark.skipif(HIPCC is None, reason="hipcc not available")

TR_READ = "ds_read_b64_tr_b16"
REG = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")


def _regs(operands: str) -> set[int]:
    out = set()
    for lo, hi, one in REG.findall(operands):
        if one:
            out.add(int(one))
        else:
            out.update(range(int(lo), int(hi) + 1))
    return out


_compiled: dict[str, str] = {}  # by source, for this module and test_asm_hazards_ring.py


def _assembly(source: str, tmp_path: Path) -> str:
    if source in _compiled:
        return _compiled[source]
    target = tmp_path / (Path(source).stem + ".s")
    cmd = [HIPCC, *build_lib.FLAGS, f"-I{build_lib.CSRC}", "--cuda-device-only", "-S",
           str(build_lib.CSRC / source), "-o", str(target)]
    result = subprocess.run(cmd, capture_output=True, text=True)
    assert result.returncode == 0, result.stderr[-2000:]
    _compiled[source] = target.read_text()
    return _compiled[source]


def _kernels(text: str) -> dict[str, list[str]]:
    """Bodies of the gemm_fast_kernel<AMODE, BMODE, PAIRED, ...> instantiations."""
    bodies, name = {}, None
    for line in text.splitlines():
        m = re.match(r"^(_ZN2ws16gemm_fast_kernelILi[01]ELi[01]ELb[01]E\w*):", line)
        if m:
            name = m.group(1)
            bodies[name] = []
        elif name is not None:
            if line.startswith(".Lfunc_end"):
                name = None
            else:
                bodies[name].append(line)
    return bodies


def _assembly_reads(body: list[str]) -> list[tuple[str, bool]]:
    """(instruction, whether it stands in inline assembly), comments and labels dropped."""
    out, inside = [], False
    for raw in body:
        text = raw.strip()
        if text.startswith((";;#ASMSTART", ";;#ASMEND")):
            inside = "START" in text
            continue
        line = text.split(";")[0].strip()
        if line and not line.endswith(":") and not line.startswith("."):
            out.append((line, inside))
    return out


def _violations(body: list[str]) -> tuple[int, list[str]]:
    pending: set[int] = set()
    reads, bad = 0, []
    for line, assembly in _assembly_reads(body):
        mnemonic, _, operands = line.partition(" ")
        if mnemonic == "s_waitcnt":
            if "lgkmcnt(0)" in operands:
                pending.clear()
            continue
        used = _regs(operands)
        if mnemonic == TR_READ or (assembly and mnemonic == "ds_read_b128"):
            reads += 1
            dest = _regs(operands.split(",")[0])
            # A second read into a pending register, or an address taken from one.
            if used & pending:
                bad.append(f"touches a pending read's register: {line}")
            pending |= dest
            continue
        if pending and mnemonic.startswith(("s_branch", "s_cbranch", "s_setpc", "s_swappc")):
            bad.append(f"branch with reads pending: {line}")
        if used & pending:
            bad.append(f"touches a pending read's register: {line}")
    if pending:
        bad.append("reads still pending at the end of the kernel")
    return reads, bad


# Instantiations per source: four operand layouts for every epilogue that runs there, the
# paired one (mm.hip) included.
@pytest.mark.parametrize("source,count", [("mm.hip", 8), ("fused.hip", 20), ("ce.hip", 24)])
def test_fragment_reads_are_waited_for_before_use(source, count, tmp_path):
    kernels = _kernels(_assembly(source, tmp_path))
    assert len(kernels) == count, (source, sorted(kernels))
    for name, body in kernels.items():
        a_mn, b_mn = re.match(r".*?ILi(\d)ELi(\d)E", name).groups()
        # A k-tile's two k32 steps read 4 A and 8 B blocks each, a transposed block in two
        # reads.
        per_tile = 2 * (4 * (1 + int(a_mn)) + 8 * (1 + int(b_mn)))
        reads, bad = _violations(body)
        assert reads >= per_tile and reads % per_tile == 0, (name, reads, per_tile)
        assert not bad, (name, bad[:5])


def test_checker_flags_a_use_before_the_wait():
    """The rule itself, on hand-written sequences: a use of a pending read's register, a
    second read into it, or a branch while reads are pending is flagged; after the wait
    the same use is clean."""
    read = "\tds_read_b64_tr_b16 v[10:11], v200 offset:512"
    mfma = "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], v[20:23], v[0:3]"
    wait = "\ts_waitcnt lgkmcnt(0)"
    assert _violations([read, wait, mfma]) == (1, [])
    assert _violations([read, mfma, wait])[1]
    assert _violations([read, "\tds_read_b64_tr_b16 v[11:12], v201", wait])[1]
    assert _violations([read, "\ts_cbranch_scc1 .LBB0_5", wait])[1]
    assert _violations([read, "\tv_add_u32_e32 v30, v31, v32", wait]) == (1, [])
    assert _violations([read])[1]
    rows = [";;#ASMSTART", "\tds_read_b128 v[20:23], v201", ";;#ASMEND"]
    assert _violations([*rows, wait, mfma]) == (1, [])
    assert _violations([*rows, mfma, wait])[1]
    assert _violations([*rows, read, wait]) == (2, [])
    assert _violations([rows[1], mfma]) == (0, [])  # the compiler's own read
