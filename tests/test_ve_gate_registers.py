"""The value-embedding gate's kernels are instantiated for each head count, and their registers grow with it: none may spill
(scratch memory), up to the 16 heads that the entry points take, by the compiler's own report for gfx950. From 13 heads a
backward that kept two rows in registers spilled and took up to three times as long."""
import re
import subprocess
import tempfile
from pathlib import Path

import pytest

from nanochat_amd import native


@pytest.fixture(scope="module")
def assembly():
    with tempfile.TemporaryDirectory() as tmp:
        out = Path(tmp) / "ve.s"
        subprocess.run([native.hipcc(), *native.HIPCC_FLAGS, f"-I{native.CSRC}", "--cuda-device-only", "-S",
                        "-o", str(out), str(native.CSRC / "ve_gate.hip")], check=True, capture_output=True)
        return out.read_text()


@pytest.mark.parametrize("kernel", ["ve_forward", "ve_backward", "ve_weight"])
def test_no_head_count_spills(assembly, kernel):
    scratch = re.findall(r"\.amdhsa_kernel _ZN2nc12_GLOBAL__N_1\d+" + kernel + r"_kernelILi(\d+)E(\w*)\n(?:.*\n)*?"
                         r"\s+\.amdhsa_private_segment_fixed_size (\d+)", assembly)
    assert {int(heads) for heads, _, _ in scratch} == set(range(1, 17))
    assert not [s for s in scratch if int(s[2])]


@pytest.mark.parametrize("heads", range(1, 17))
def test_weight_gradient_runs_in_one_round(assembly, lib, heads):
    """Its slabs of rows, by the workspace they need, times the column chunks are no more workgroups (four waves, one a
    SIMD) than the registers let run at once on 256 CUs: a second round would be nearly empty."""
    used = int(re.search(r"\.amdhsa_kernel _ZN2nc12_GLOBAL__N_116ve_weight_kernelILi%dE\w*\n(?:.*\n)*?"
                         r"\s+\.amdhsa_next_free_vgpr (\d+)" % heads, assembly).group(1))
    resident = 256 * min(8, 512 // (-(-used // 8) * 8))
    for rows in (4096, 16384, 65536):
        slabs = lib.nc_ve_weight_grad_workspace_bytes(rows, heads) // (heads * heads * 128 * 4)
        assert slabs * (-(-heads // 2)) <= resident
