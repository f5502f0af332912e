// Instantiations of the fp16 GEMM whose workgroups stay for several tiles, compiled to assembly by
// tests/test_isa_hazards_gemm_wide.py (never linked, never run).
#include "../../daceml_amd/csrc/gemm_f16_wide.h"

namespace dml {
namespace gemm16 {

const void* wide_gemm_kernels[] = {
    // blocks of a wavefront in either direction, A kind, B kind, epilogue, K-concatenated pairs, K in slices
    (const void*)gemm_f16_wide_kernel<8, 0, 0, EPI_PLAIN, false>, (const void*)gemm_f16_wide_kernel<8, 0, 0, EPI_GENERAL, false>,
    (const void*)gemm_f16_wide_kernel<8, 1, 1, EPI_PLAIN, false>, (const void*)gemm_f16_wide_kernel<8, 0, 1, EPI_GENERAL, true>,
    (const void*)gemm_f16_wide_kernel<8, 1, 1, EPI_PLAIN, false, true>,
    (const void*)gemm_f16_wide_kernel<4, 0, 0, EPI_GENERAL, false>, (const void*)gemm_f16_wide_kernel<4, 0, 1, EPI_GENERAL, true>};

}  // namespace gemm16
}  // namespace dml
