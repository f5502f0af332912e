// Launches the fp16 GEMM of gemm_f16_wide.h: tile configuration 13.
#include "gemm_f16_wide.h"

namespace dml {
namespace gemm16 {

namespace {
template <int AKIND, int BKIND, int EPI, bool KSUM>
int launch(const GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* residual,
           hipStream_t st) {
    auto kern = gemm_f16_wide_kernel<AKIND, BKIND, EPI, KSUM>;
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kWideLds);
    if (e != hipSuccess) {
        set_error("gemm_f16: cannot reserve %d bytes of LDS: %s", kWideLds, hipGetErrorString(e));
        return (int)e;
    }
    const unsigned grid = (unsigned)(g.total_blocks < kCus ? g.total_blocks : kCus);
    hipLaunchKernelGGL(kern, grid, kThreads, kWideLds, st, a, b, c, bias, residual, g);
    return launch_status("gemm_f16(wide)");
}
}  // namespace

int launch_wide(GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* residual, int ak, int bk, long long batch, hipStream_t st) {
    g.tiles_m = (g.m + kWideTile - 1) / kWideTile;
    g.tiles_n = (g.n + kWideTile - 1) / kWideTile;
    const long long total = (long long)g.tiles_m * g.tiles_n * batch;
    DML_REQUIRE(total <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f16: %lld workgroups exceed the grid limit", total);
    g.total_blocks = total;
    const int ek = epilogue_kind(g, bias, residual, nullptr);
#define DML_WIDE_CASE(AK, BKD, EPI, KSUM)                   \
    if (ak == AK && bk == BKD && ek == EPI && !!g.ksum == KSUM) \
        return launch<AK, BKD, EPI, KSUM>(g, a, b, c, bias, residual, st);
#define DML_WIDE_CASES(EPI, KSUM) \
    DML_WIDE_CASE(0, 0, EPI, KSUM) DML_WIDE_CASE(0, 1, EPI, KSUM) DML_WIDE_CASE(1, 0, EPI, KSUM) DML_WIDE_CASE(1, 1, EPI, KSUM)
    DML_WIDE_CASES(EPI_PLAIN, false) DML_WIDE_CASES(EPI_GENERAL, false)
    DML_WIDE_CASES(EPI_PLAIN, true) DML_WIDE_CASES(EPI_GENERAL, true)
#undef DML_WIDE_CASES
#undef DML_WIDE_CASE
    set_error("gemm_f16: no 256 x 256 kernel for operand kinds %d/%d, epilogue %d", ak, bk, ek);
    return DMLHIP_ERR_UNSUPPORTED;
}

}  // namespace gemm16
}  // namespace dml
