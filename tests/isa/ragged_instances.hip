// The pipelined GEMM kernel with a ragged last K step, one instance per tile configuration with and without row sums,
// compiled to assembly by tests/test_isa_hazards.py (never linked, never run).
#include "../../daceml_amd/csrc/gemm_f16_pipe.h"

namespace dml {
namespace gemm16 {

#define RAGGED_KERNEL(BM, BN, WM, WN, NSTAGE, ASUM) \
    (const void*)gemm_f16_pipe_kernel<BM, BN, WM, WN, 1, 1, NSTAGE, EPI_PLAIN, false, ASUM, true, true>

const void* isa_check_kernels[] = {
    RAGGED_KERNEL(256, 256, 128, 128, 2, false), RAGGED_KERNEL(128, 128, 64, 64, 4, false),
    RAGGED_KERNEL(128, 128, 64, 64, 2, false),   RAGGED_KERNEL(128, 64, 64, 32, 3, false),
    RAGGED_KERNEL(128, 128, 64, 64, 4, true),    RAGGED_KERNEL(128, 128, 64, 64, 2, true)};

}  // namespace gemm16
}  // namespace dml
