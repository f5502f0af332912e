// Launches the 256 x 256 tile of gemm_f16_wide.h (configuration 13) and the weight gradients in slices.
#include "gemm_f16_wide.h"

namespace dml {
namespace gemm16 {

int launch_wide256(GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* residual, int ak,
                   int bk, long long batch, hipStream_t st) {
    DML_WIDE_TILES(8)
    DML_WIDE_CASES(8, 0, 0) DML_WIDE_CASES(8, 0, 1) DML_WIDE_CASES(8, 1, 0) DML_WIDE_CASES(8, 1, 1)
    return wide_unsupported(ak, bk);
}

size_t wide_sliced_bytes(int64_t m, int64_t n, int groups, int slices, size_t* row_offset) {
    const size_t results = (size_t)groups * slices * m * n * sizeof(float);
    *row_offset = (results + 255) & ~(size_t)255;
    return *row_offset + (size_t)groups * slices * ceil_div(n, (int64_t)kWideTile) * 2 * m * sizeof(float);
}

int launch_wide_sliced(GemmArgs& g, int groups, int slices, const _Float16* const* a, const _Float16* const* b, void* const* c,
                       void* const* asum, int asum_f32, int bk, void* workspace, hipStream_t st) {
    size_t row_offset;
    wide_sliced_bytes(g.m, g.n, groups, slices, &row_offset);
    WideSumArgs sum{};
    sum.part = reinterpret_cast<const float*>(workspace);
    sum.row_part = reinterpret_cast<const float*>(reinterpret_cast<const char*>(workspace) + row_offset);
    sum.slices = slices;
    sum.count = (int64_t)g.m * g.n;
    sum.m = g.m;
    sum.out_f32 = g.out_f32;
    sum.asum_f32 = asum_f32;
    sum.alpha = g.alpha;
    g.tiles_m = (g.m + kWideTile - 1) / kWideTile;
    g.tiles_n = (g.n + kWideTile - 1) / kWideTile;
    sum.row_parts = slices * g.tiles_n * 2;
    g.groups = groups;
    g.ksum = 0;
    g.batch1 = slices;
    g.batch2 = 1;
    for (int i = 0; i < 3; ++i) g.sab[i] = g.sbb[i] = g.scb[i] = 0;
    g.scb[1] = sum.count;
    g.scm = g.n;
    g.alpha = 1.f;
    g.out_f32 = 1;
    g.asum = asum ? const_cast<float*>(sum.row_part) : nullptr;
    for (int i = 0; i < groups; ++i) {
        g.ga[i] = a[i];
        g.gb[i] = b[i];
        g.gc[i] = const_cast<float*>(sum.part) + (int64_t)i * slices * sum.count;
        g.gbias[i] = nullptr;
        sum.out[i] = c[i];
        sum.asum[i] = asum ? asum[i] : nullptr;
    }
    g.total_blocks = (long long)g.tiles_m * g.tiles_n * groups * slices;
    const int e = bk == 0 ? launch_shape<8, 1, 0, EPI_PLAIN, false, true>(g, a[0], b[0], g.gc[0], nullptr, nullptr, st)
                          : launch_shape<8, 1, 1, EPI_PLAIN, false, true>(g, a[0], b[0], g.gc[0], nullptr, nullptr, st);
    if (e) return e;
    const int blocks = (int)ceil_div(sum.count, (int64_t)1024);
    const dim3 grid(blocks + (asum ? (g.m + 63) / 64 : 0), groups);
    hipLaunchKernelGGL(wide_sum_kernel, grid, 256, 0, st, sum, blocks);
    return launch_status("gemm_f16(sum of slices)");
}

}  // namespace gemm16
}  // namespace dml
