"""No instruction of the split 3 x 3 weight gradient touches a register that an LDS read in flight still has to write."""
import os

from tests import isa_hazards
from tests.test_isa_hazards import ROOT, _assembly, _kernel_count, _report


def test_split_weight_gradient(tmp_path):
    asm = _assembly(os.path.join(ROOT, "daceml_amd", "csrc", "conv_dense3_weight_split.hip"), tmp_path)
    assert _kernel_count(asm, "conv_dense3_weight_split_kernel") == 8
    found = isa_hazards.check_file(asm)[1]
    assert not found, _report(found)
