"""No instruction of the fp16 GEMM with tiles that stay touches a register that an LDS read in flight still has to write."""
import os

from tests import isa_hazards
from tests.test_isa_hazards import ROOT, _assembly, _kernel_count, _report


def test_wide_gemm(tmp_path):
    asm = _assembly(os.path.join(ROOT, "tests", "isa", "wide_instances.hip"), tmp_path)
    assert _kernel_count(asm, "gemm_f16_wide_kernel") == 7
    found = isa_hazards.check_file(asm)[1]
    assert not found, _report(found)
    # the accumulators stay where they are, and nothing of the loop goes through memory
    text = open(asm).read()
    assert "scratch_" not in text and "v_accvgpr_mov" not in text and "v_accvgpr_write" not in text
