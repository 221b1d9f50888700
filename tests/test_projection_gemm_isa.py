"""The projection GEMM (prefill_gemm.hip's tiles with the residual and row-statistic epilogue) keeps the MFMA hazards by
the same construction as the prefill GEMM; the same checks on its gfx950 assembly. And for both: the LDS reads are inline
assembly, whose results the compiler takes as written at once, so nothing may read or write a read's registers before an
s_waitcnt lgkmcnt(0) has let it land, on any path."""
import re
import subprocess
import tempfile
from pathlib import Path

import pytest

from nanochat_amd import native
from tests.test_prefill_gemm_isa import (SOURCE, blocks, loop_lines, mfma_operand_writers, regs,
                                         wait_states_before_agpr_reads)

MODES = (0, 1, 2)   # whole tiles, split, thin


def early_uses(lines):
    """The instructions that touch a register a ds_read has yet to fill: a forward fixed point over the basic blocks of
    the registers pending on some path. Writing one is as wrong as reading it (the read lands later)."""
    bl = blocks(lines)
    index = {lab: i for i, (lab, _, _) in enumerate(bl)}
    state_in, work, found = {0: frozenset()}, [0], set()
    while work:
        i = work.pop()
        pending = set(state_in[i])
        for n, (mn, ops) in enumerate(bl[i][1]):
            if mn == "s_waitcnt":
                text = " ".join(ops)
                if "lgkmcnt(0)" in text or not text.strip("0x "):
                    pending = set()
                continue
            touched = set().union(*(regs(op) for op in ops)) if ops else set()
            if touched & pending:
                found.add((bl[i][0], n, mn, tuple(ops)))
            if mn.startswith("ds_read"):
                pending |= regs(ops[0])
        for t in bl[i][2]:
            k = index[t]
            new = state_in.get(k, frozenset()) | pending
            if k not in state_in or new != state_in[k]:
                state_in[k] = new
                work.append(k)
    return sorted(found)


def test_early_uses_are_seen():
    late = """
        ds_read_b128 v[0:3], v20
        v_add_u32_e32 v9, v8, v7
        s_waitcnt lgkmcnt(0)
        v_add_u32_e32 v2, v8, v7
        s_endpgm
    """.splitlines()
    assert not early_uses(late)
    early = [l for l in late if "s_waitcnt" not in l]
    assert [e[2:] for e in early_uses(early)] == [("v_add_u32_e32", ("v2", "v8", "v7"))]


@pytest.fixture(scope="module")
def assembly():
    with tempfile.TemporaryDirectory() as tmp:
        out = Path(tmp) / "pg.s"
        subprocess.run([native.hipcc(), *native.HIPCC_FLAGS, f"-I{native.CSRC}", "--cuda-device-only", "-S",
                        "-o", str(out), str(SOURCE)], check=True, capture_output=True)
        return out.read_text()


def bodies(text, name):
    return {m.group(1): m.group(2).splitlines() for m in re.finditer(
        r"^(_ZN2nc\d+" + name + r"_kernelI\w*):[^\n]*\n(.*?)\n\.Lfunc_end", text, re.S | re.M)}


def test_nothing_touches_a_read_in_flight(assembly):
    found = {**bodies(assembly, "prefill_gemm"), **bodies(assembly, "projection_gemm")}
    assert len(found) == 15
    for name, lines in found.items():
        assert not early_uses(lines), (name, early_uses(lines)[:4])


@pytest.fixture(scope="module")
def kernels(assembly):
    return {int(m.group(1)): m.group(2).splitlines() for m in re.finditer(
        r"^_ZN2nc22projection_gemm_kernelILi([012])EEEvNS_6PfGemmE\w*:[^\n]*\n(.*?)\n\.Lfunc_end", assembly, re.S | re.M)}


@pytest.mark.parametrize("mode", MODES)
def test_hazards_kept(kernels, mode):
    assert sorted(kernels) == list(MODES)
    found = mfma_operand_writers(kernels[mode])
    assert len(found) >= 32
    assert all(kinds == {"ds_read"} for kinds in found.values())
    assert not any("v_accvgpr" in l for l in loop_lines(kernels[mode]))
    assert not any("scratch_" in l for l in kernels[mode])
    assert wait_states_before_agpr_reads(kernels[mode]) >= 32
