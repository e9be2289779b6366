"""The rule of test_asm_hazards.py on the smaller macro-tiles' kernel (CPU only): with an
M/N-contiguous operand all of its k-loop's fragment reads are inline assembly, the
transposing ones and, for a K-contiguous operand beside it, ``ds_read_b128``. No
instruction may touch a pending read's destination, and no branch may leave with one
pending, before the next ``s_waitcnt lgkmcnt(0)``."""
import re

import pytest

from test_asm_hazards import HIPCC, TR_READ, _assembly, _regs

pytestmark = pytest.mark.skipif(HIPCC is None, reason="hipcc not available")


def _ring_kernels(text: str) -> dict[str, list[str]]:
    """Bodies of the gemm_ring_kernel<RingCfg, AMODE, BMODE, ...> instantiations with an
    M/N-contiguous operand."""
    bodies, name = {}, None
    for line in text.splitlines():
        m = re.match(r"^(_ZN2ws16gemm_ring_kernelINS_7RingCfg\w+?EEELi(\d)ELi(\d)E\w*):", line)
        if m:
            name = m.group(1) if "1" in m.group(2, 3) else None
            if name:
                bodies[name] = []
        elif name is not None:
            if line.startswith(".Lfunc_end"):
                name = None
            else:
                bodies[name].append(line.split(";")[0].strip())
    return bodies


def _violations(body: list[str]) -> tuple[int, list[str]]:
    reads = [i for i, line in enumerate(body) if line.startswith(TR_READ)]
    pending, bad = set(), []
    # From the first transposing read's group to the loop's last wait: a K-contiguous
    # operand's reads precede or follow the transposing ones without a branch between.
    first = max((i for i in range(reads[0]) if body[i].startswith(("s_barrier", ".LBB"))), default=0)
    last = next(i for i in range(reads[-1], len(body))
                if body[i].startswith("s_waitcnt") and "lgkmcnt(0)" in body[i])
    for line in body[first:last + 1]:
        mnemonic, _, operands = line.partition(" ")
        if mnemonic == "s_waitcnt":
            if "lgkmcnt(0)" in operands:
                pending.clear()
            continue
        if not line or line.startswith(".") or line.endswith(":"):
            continue
        if mnemonic in (TR_READ, "ds_read_b128"):
            dest = _regs(operands.split(",")[0])
            if dest & pending:
                bad.append(f"overwrites a pending read's register: {line}")
            pending |= dest
            continue
        if pending and mnemonic.startswith(("s_branch", "s_cbranch", "s_setpc", "s_swappc")):
            bad.append(f"branch with reads pending: {line}")
        if _regs(operands) & pending:
            bad.append(f"touches a pending read's register: {line}")
    if pending:
        bad.append("reads still pending after the last wait")
    return len(reads), bad


@pytest.mark.parametrize("source", ["mm.hip", "fused.hip"])
def test_ring_reads_are_waited_for_before_use(source, tmp_path):
    kernels = _ring_kernels(_assembly(source, tmp_path))
    assert kernels, f"no ring instantiation with an M/N-contiguous operand in {source}"
    for name, body in kernels.items():
        reads, bad = _violations(body)
        assert reads >= 8, (name, reads)  # two blocks, two reads each, two k32 steps
        assert not bad, (name, bad[:5])


def test_checker_flags_a_use_before_the_wait():
    tr, rows = f"{TR_READ} v[10:11], v200", "ds_read_b128 v[20:23], v201"
    mfma = "v_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], v[20:23], v[0:3]"
    wait = "s_waitcnt lgkmcnt(0)"
    assert _violations(["s_barrier", rows, tr, wait, mfma]) == (1, [])
    assert _violations(["s_barrier", rows, tr, mfma, wait])[1]
    assert _violations(["s_barrier", rows, "v_add_u32_e32 v20, v1, v2", tr, wait])[1]
    assert _violations(["s_barrier", tr, "s_cbranch_scc1 .LBB0_5", wait])[1]
