"""The assembly of the fp16 GEMM with tiles that stay, every instantiation that the library launches: no instruction touches a
register that an LDS read in flight still has to write, and the matrix instructions, which are inline assembly, have the wait
states that the compiler does not keep for them."""
import os
import re

import pytest

from tests import isa_hazards
from tests.test_isa_hazards import ROOT, _assembly, _kernel_count, _report


@pytest.mark.parametrize("source,count", [("gemm_f16_wide.hip", 18), ("gemm_f16_wide_half.hip", 8)])
def test_wide_gemm(source, count, tmp_path):
    """256 x 256 tiles: four operand layouts, two epilogues, with and without operand pairs, and two kernels of slices; 128 x 128
    tiles: two layouts."""
    asm = _assembly(os.path.join(ROOT, "daceml_amd", "csrc", source), tmp_path)
    assert _kernel_count(asm, "gemm_f16_wide_kernel") == count
    found = isa_hazards.check_file(asm)[1]
    assert not found, _report(found)
    assert not isa_hazards.check_mfma(asm)
    # the accumulators stay where they are, and nothing goes through memory where matrix instructions are issued (two of the kernels
    # with both operands row-contiguous keep an address there across the loop)
    for name, body in isa_hazards.kernels(asm):
        for block in _blocks(body):
            assert not any(code.startswith(("v_accvgpr_mov", "v_accvgpr_write")) for code in block), name
            if any(code.startswith("v_mfma") for code in block):
                assert not any(code.startswith("scratch_") for code in block), name


def _blocks(body):
    block = []
    for _, kind, code in body:
        if kind == "label" or re.match(r"s_c?branch|s_endpgm", code):
            yield block
            block = []
        else:
            block.append(code)
    yield block


def test_the_check_of_matrix_instructions_finds_what_it_is_for(tmp_path):
    text = """
_Z6kernelv:
	v_mov_b32_e32 v9, 0
	s_nop 1
	v_mfma_f32_16x16x32_f16 a[0:3], v[8:11], v[4:7], a[0:3]
	s_nop 15
	s_nop 1
	v_accvgpr_read_b32 v1, a3
	s_endpgm
.Lfunc_end0:
"""
    p = tmp_path / "k.s"
    p.write_text(text)
    assert not isa_hazards.check_mfma(str(p))
    for was, now, line in (("\ts_nop 1\n\tv_mfma", "\ts_nop 0\n\tv_mfma", 5), ("\ts_nop 1\n\tv_mfma", "\tv_mfma", 4),
                           ("\ts_nop 1\n\tv_accvgpr", "\ts_nop 0\n\tv_accvgpr", 8)):
        p.write_text(text.replace(was, now))
        assert sorted(isa_hazards.check_mfma(str(p))["_Z6kernelv"]) == [line]
