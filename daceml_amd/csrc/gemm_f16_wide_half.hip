// Launches the 128 x 128 tile of gemm_f16_wide.h (configuration 14), for a K-contiguous A: a translation unit of its own so that
// it compiles beside the other.
#include "gemm_f16_wide.h"

namespace dml {
namespace gemm16 {

int launch_wide128(GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* residual, int ak,
                   int bk, long long batch, hipStream_t st) {
    DML_WIDE_TILES(4)
    DML_WIDE_CASES(4, 0, 0) DML_WIDE_CASES(4, 0, 1)
    return wide_unsupported(ak, bk);
}

}  // namespace gemm16
}  // namespace dml
