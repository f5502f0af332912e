// The pipelined fp16 GEMM kernel for a K that is no multiple of 64, in the tile configurations of the weight gradients
// (both operands row-contiguous, K = tokens): a translation unit of its own so that it compiles beside the others.
#include "gemm_f16_pipe.h"

namespace dml {
namespace gemm16 {

int launch_pipelined_ragged(GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* residual,
                            void* pre, int cfg, long long batch, hipStream_t st) {
    if (g.asum || (g.groups && g.gasum[0])) {
        if (cfg == 7) return launch_tile<128, 128, 64, 64, 2, false, true, true, true>(g, a, b, c, bias, residual, pre, 1, 1, batch, st);
        return launch_tile<128, 128, 64, 64, 4, false, true, true, true>(g, a, b, c, bias, residual, pre, 1, 1, batch, st);
    }
    switch (cfg) {
        case 4: return launch_tile<256, 256, 128, 128, 2, false, false, true, true>(g, a, b, c, bias, residual, pre, 1, 1, batch, st);
        case 7: return launch_tile<128, 128, 64, 64, 2, false, false, true, true>(g, a, b, c, bias, residual, pre, 1, 1, batch, st);
        case 9: return launch_tile<128, 64, 64, 32, 3, false, false, true, true>(g, a, b, c, bias, residual, pre, 1, 1, batch, st);
        default: return launch_tile<128, 128, 64, 64, 4, false, false, true, true>(g, a, b, c, bias, residual, pre, 1, 1, batch, st);
    }
}

}  // namespace gemm16
}  // namespace dml
