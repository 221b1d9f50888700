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
