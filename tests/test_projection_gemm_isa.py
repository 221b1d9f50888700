"""The projection GEMM (prefill_gemm.hip's tiles with the residual and row-statistic epilogue) keeps the MFMA hazards by
the same construction as the prefill GEMM; the same checks on its gfx950 assembly."""
import re
import subprocess
import tempfile
from pathlib import Path

import pytest

from nanochat_amd import native
from tests.test_prefill_gemm_isa import SOURCE, loop_lines, mfma_operand_writers, wait_states_before_agpr_reads

MODES = (0, 1, 2)   # whole tiles, split, thin


@pytest.fixture(scope="module")
def kernels():
    with tempfile.TemporaryDirectory() as tmp:
        out = Path(tmp) / "pg.s"
        subprocess.run([native.hipcc(), *native.HIPCC_FLAGS, f"-I{native.CSRC}", "--cuda-device-only", "-S",
                        "-o", str(out), str(SOURCE)], check=True, capture_output=True)
        text = out.read_text()
    return {int(m.group(1)): m.group(2).splitlines() for m in re.finditer(
        r"^_ZN2nc22projection_gemm_kernelILi([012])EEEvNS_6PfGemmE\w*:[^\n]*\n(.*?)\n\.Lfunc_end", text, re.S | re.M)}


@pytest.mark.parametrize("mode", MODES)
def test_hazards_kept(kernels, mode):
    assert sorted(kernels) == list(MODES)
    found = mfma_operand_writers(kernels[mode])
    assert len(found) >= 32
    assert all(kinds == {"ds_read"} for kinds in found.values())
    assert not any("v_accvgpr" in l for l in loop_lines(kernels[mode]))
    assert not any("scratch_" in l for l in kernels[mode])
    assert wait_states_before_agpr_reads(kernels[mode]) >= 32
