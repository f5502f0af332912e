// The instantiations of the GEMM kernels that one step of the benchmarked BERT layer launches, and those of the pipelined kernel
// that such products are on where they fill the chip less (the fused expand + depthwise kernels and the attention kernels are
// taken from their own source files), compiled to assembly by tests/test_validated_kernels.py (never linked, never run) and
// compared with the instruction digests recorded when these kernels last passed their tests on the GPU.
#include "../../daceml_amd/csrc/gemm_f16_pipe.h"
#include "../../daceml_amd/csrc/gemm_f16_wide.h"

namespace dml {
namespace gemm16 {

const void* validated_gemm_kernels[] = {
    // BM, BN, WM, WN, A kind, B kind, stages, epilogue, K-concatenated pairs, row sums, interleaved loop
    (const void*)gemm_f16_pipe_kernel<128, 128, 64, 64, 1, 1, 4, EPI_PLAIN, false, true, true>,      // the step's weight + bias gradients
    (const void*)gemm_f16_pipe_kernel<128, 128, 64, 64, 0, 0, 4, EPI_PLAIN, false, false, true>,
    (const void*)gemm_f16_pipe_kernel<128, 128, 64, 64, 0, 0, 4, EPI_GENERAL, false, false, true>,
    (const void*)gemm_f16_pipe_kernel<256, 256, 128, 128, 0, 0, 2, EPI_PLAIN, false, false, true>,
    (const void*)gemm_f16_pipe_kernel<256, 256, 128, 128, 0, 1, 2, EPI_PLAIN, false, false, true>,
    (const void*)gemm_f16_pipe_kernel<128, 128, 64, 64, 0, 1, 4, EPI_GENERAL, false, false, true>,
    (const void*)gemm_f16_pipe_kernel<128, 128, 64, 64, 0, 1, 4, EPI_GENERAL, true, false, true>,
    (const void*)gemm_f16_pipe_kernel<128, 128, 64, 64, 0, 1, 4, EPI_PLAIN, false, false, true>,     // the step's o input gradient
    (const void*)gemm_f16_pipe_kernel<128, 64, 64, 32, 0, 0, 3, EPI_PLAIN, false, false, true>,      // few tiles, long K
    // blocks of a wavefront, A kind, B kind, epilogue, K-concatenated pairs. The step's
    (const void*)gemm_f16_wide_kernel<8, 0, 0, EPI_PLAIN, false>,     // q/k/v projections (grouped), FFN1
    (const void*)gemm_f16_wide_kernel<4, 0, 0, EPI_GENERAL, false>,   // o and FFN2 with residual
    (const void*)gemm_f16_wide_kernel<8, 0, 1, EPI_PLAIN, false>,     // FFN2 input gradient
    (const void*)gemm_f16_wide_kernel<4, 0, 1, EPI_GENERAL, false>,   // FFN1 input gradient with residual
    (const void*)gemm_f16_wide_kernel<4, 0, 1, EPI_GENERAL, true>};   // q/k/v input gradients summed

}  // namespace gemm16
}  // namespace dml
