// 1x1 convolutions of few input and many output channels, fp32 (the expansion of an inverted-residual block, and the data
// gradient of its projection): Y[n, m, p] = act(sum_c W[m, c] X[n, c, p] + b[m]).
//
// What bounds them: the write of Y; with at most 48 input channels the product has one or two K steps, and a tiled GEMM
// spends its time on filling and draining a ring per tile (and on rows of a last tile that is half empty). Here a wavefront
// takes 32 pixels and keeps all their input channels in registers - one 4-byte load per channel and lane, all in flight at
// once, no alignment needed - and multiplies them on v_mfma_f32_32x32x2_f32 with block after block of 32 output channels,
// whose weights a workgroup has in LDS. Rows of Y leave in pieces of 128 bytes while the next block is multiplied.
// Pixels are counted through the batch; with few of them the output channels are split over the grid.
// Measured, us, forward / data gradient of the mirrored convolution: 24 -> 144 channels, 32 x 56 x 56, 36.4 / 30.4 (tiled
// GEMM / streaming kernel; the others beside an older GEMM), 24.9 / 24.1 a float at a time and 16.7 / 15.9 in fours
// (67 MB, 4.1 TB/s), 55 x 55 56 / 54 and 22.6 / 21.5,
// 16 -> 96, 32 x 112 x 112, 97 / 58, 32.5 / 33.2 and 31.3 / 29.8 (180 MB, 5.9 TB/s), 40 -> 240, 32 x 28 x 28, 29 / 32, 16.9 / 15.7 and 12.8 / 13.2,
// 40 -> 240, 2 x 28 x 28, 22 / 19, 5.2 / 5.0 and 4.2 / 4.3. 32 -> 192, 32 x 56 x 56, stays with
// the streaming kernel forward (32 us there, 38 here) and comes here for the data gradient (45 there, 33 here).
#include "common.h"
#include "conv_geom.h"

#include <type_traits>

namespace dml {
namespace {

constexpr int kFewWaves = 4;
constexpr int kFewMaxIn = 48;
constexpr int kFewVecBlocks = 9;   // blocks of 16 output channels per workgroup, at most
constexpr int kFewBlocks = 8;      // blocks of 32 output channels per workgroup, at most: 48 KB of weights

struct FewArgs {
    const float* x;
    const float* w;
    const float* bias;
    float* y;
    int cin, cout, act;
    uint32_t hw, pixels;           // of an image, of all
    int blocks;                    // blocks of 32 output channels per workgroup
};

// KP: pairs of input channels. WT: w is [cin][cout].
template <int KP, bool WT>
__global__ __launch_bounds__(64 * kFewWaves) void conv_pointwise_few_kernel(const FewArgs g) {
    // [input channel][output channel]: the two halves of a wavefront read 32 floats each of neighbouring rows
    __shared__ float ws[2 * KP * kFewBlocks * 32 + kFewBlocks * 32];
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    const uint32_t p = (blockIdx.x * kFewWaves + threadIdx.x / 64) * 32u + l32;
    const bool ok = p < g.pixels;
    const uint32_t pc = ok ? p : g.pixels - 1, n = pc / g.hw;      // behind the end: a pixel that is there, not stored
    const float* x = g.x + (size_t)n * g.cin * g.hw + (pc - n * g.hw);
    float b[KP];
#pragma unroll
    for (int k = 0; k < KP; ++k) b[k] = x[(size_t)min(2 * k + h, g.cin - 1) * g.hw];
    const int m0 = blockIdx.y * g.blocks * 32, rows = g.blocks * 32;
    float* bs = ws + 2 * KP * rows;
    // consecutive threads read along the weights' rows, eight loads each before the first is stored
    const int count = 2 * KP * rows;
    for (int i0 = threadIdx.x; i0 < count; i0 += 64 * kFewWaves * 8) {
        float v[8];
        int at[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(i0 + u * 64 * kFewWaves, count - 1);   // behind the end: the last one again
            const int c = WT ? i / rows : i % (2 * KP), m = WT ? i - c * rows : i / (2 * KP);
            const bool in = c < g.cin && m0 + m < g.cout;
            at[u] = c * rows + m;
            v[u] = g.w[!in ? 0 : WT ? (size_t)c * g.cout + m0 + m : (size_t)(m0 + m) * g.cin + c];
            v[u] = in ? v[u] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) ws[at[u]] = v[u];
    }
    for (int i = threadIdx.x; i < rows; i += 64 * kFewWaves) bs[i] = g.bias && m0 + i < g.cout ? g.bias[m0 + i] : 0.f;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KP; ++k) b[k] = 2 * k + h < g.cin ? b[k] : 0.f;
    float* y = g.y + (size_t)n * g.cout * g.hw + (pc - n * g.hw);
    auto all = [&](auto actc) {
        constexpr int ACT = decltype(actc)::value;
        for (int i = 0; i < rows && m0 + i < g.cout; i += 32) {
            floatx16 acc;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = bs[i + (e >> 2) * 8 + h * 4 + (e & 3)];
#pragma unroll
            for (int k = 0; k < KP; ++k)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ws[(2 * k + h) * rows + i + l32], b[k], acc, 0, 0, 0);
            if (!ok) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + i + (e >> 2) * 8 + h * 4 + (e & 3);
                if (m < g.cout) y[(size_t)m * g.hw] = apply_act(ACT, acc[e]);
            }
        }
    };
    switch (g.act) {
        case DMLHIP_ACT_GELU: all(std::integral_constant<int, DMLHIP_ACT_GELU>{}); break;
        case DMLHIP_ACT_SWISH: all(std::integral_constant<int, DMLHIP_ACT_SWISH>{}); break;
        case DMLHIP_ACT_SIGMOID: all(std::integral_constant<int, DMLHIP_ACT_SIGMOID>{}); break;
        case DMLHIP_ACT_RELU: all(std::integral_constant<int, DMLHIP_ACT_RELU>{}); break;
        default: all(std::integral_constant<int, DMLHIP_ACT_NONE>{}); break;
    }
}

// The same for images whose pixels can be read in fours: 64 pixels per wavefront on v_mfma_f32_16x16x4_f32, four consecutive ones
// per lane, so that X is read and Y written sixteen bytes per lane and 256 bytes in a row. KS: steps of four input channels.
template <int KS, bool WT>
__global__ __launch_bounds__(64 * kFewWaves) void conv_pointwise_few_vec_kernel(const FewArgs g) {
    __shared__ float ws[4 * KS * (kFewVecBlocks * 16 + 16) + kFewVecBlocks * 16];
    const int lane = threadIdx.x & 63, q = lane & 15, kk = lane >> 4;
    const uint32_t p = (blockIdx.x * kFewWaves + threadIdx.x / 64) * 64u + 4u * q;
    const bool ok = p < g.pixels;
    const uint32_t pc = ok ? p : g.pixels - 4, n = pc / g.hw;      // behind the end: pixels that are there, not stored
    const float* x = g.x + (size_t)n * g.cin * g.hw + (pc - n * g.hw);
    floatx4 b[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) b[s] = *reinterpret_cast<const floatx4*>(x + (size_t)min(4 * s + kk, g.cin - 1) * g.hw);
    const int rows = g.blocks * 16, m0 = blockIdx.y * rows, pitch = rows | 16;   // rows of four channels: different quarters of the banks
    float* bs = ws + 4 * KS * pitch;
    const int count = 4 * KS * rows;
    for (int i0 = threadIdx.x; i0 < count; i0 += 64 * kFewWaves * 8) {
        float v[8];
        int at[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = min(i0 + u * 64 * kFewWaves, count - 1);
            const int c = WT ? i / rows : i % (4 * KS), m = WT ? i - c * rows : i / (4 * KS);
            const bool in = c < g.cin && m0 + m < g.cout;
            at[u] = c * pitch + m;
            v[u] = g.w[!in ? 0 : WT ? (size_t)c * g.cout + m0 + m : (size_t)(m0 + m) * g.cin + c];
            v[u] = in ? v[u] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) ws[at[u]] = v[u];
    }
    for (int i = threadIdx.x; i < rows; i += 64 * kFewWaves) bs[i] = g.bias && m0 + i < g.cout ? g.bias[m0 + i] : 0.f;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < KS; ++s) b[s] = 4 * s + kk < g.cin ? b[s] : floatx4{0.f, 0.f, 0.f, 0.f};
    float* y = g.y + (size_t)n * g.cout * g.hw + (pc - n * g.hw);
    auto all = [&](auto actc) {
        constexpr int ACT = decltype(actc)::value;
        for (int i = 0; i < rows && m0 + i < g.cout; i += 16) {
            floatx4 acc[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = *reinterpret_cast<const floatx4*>(bs + i + 4 * kk);
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const float a = ws[(4 * s + kk) * pitch + i + q];
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[s][j], acc[j], 0, 0, 0);
            }
            if (!ok) continue;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = m0 + i + 4 * kk + e;
                if (m < g.cout)
                    *reinterpret_cast<floatx4*>(y + (size_t)m * g.hw) =
                        floatx4{apply_act(ACT, acc[0][e]), apply_act(ACT, acc[1][e]), apply_act(ACT, acc[2][e]), apply_act(ACT, acc[3][e])};
            }
        }
    };
    switch (g.act) {
        case DMLHIP_ACT_GELU: all(std::integral_constant<int, DMLHIP_ACT_GELU>{}); break;
        case DMLHIP_ACT_SWISH: all(std::integral_constant<int, DMLHIP_ACT_SWISH>{}); break;
        case DMLHIP_ACT_SIGMOID: all(std::integral_constant<int, DMLHIP_ACT_SIGMOID>{}); break;
        case DMLHIP_ACT_RELU: all(std::integral_constant<int, DMLHIP_ACT_RELU>{}); break;
        default: all(std::integral_constant<int, DMLHIP_ACT_NONE>{}); break;
    }
}

}  // namespace

// Few input channels, at least twice as many output channels (otherwise reading X counts as much as writing Y). Over 782
// problems of 1 - 48 input and 2 - 6 times (at least 32) as many output channels, 1 - 32 images of 6 x 6 to 112 x 112, forward and data
// gradient of the mirrored convolution, none took longer than with the kernels before: 0.27 of their time in the median, at 1 : 2
// 0.95 (24 -> 48, 32 x 56 x 56).
bool pointwise_few_applicable(int64_t n, int64_t cin, int64_t cout, int64_t hw) {
    return cin >= 1 && cin <= kFewMaxIn && cout >= 2 * cin && cout >= 32 && hw >= 32 && n * hw <= 0x7fffffff - 127 &&
           cout <= 65535 * 32;
}

int launch_pointwise_few(const float* x, const float* w, const float* bias, float* y, int n, int cin, int cout, int64_t hw,
                         int act, bool w_transposed, hipStream_t st) {
    FewArgs g;
    g.x = x; g.w = w; g.bias = bias; g.y = y;
    g.cin = cin; g.cout = cout; g.act = act;
    g.hw = (uint32_t)hw;
    g.pixels = (uint32_t)(n * hw);
    // In fours wherever they can be read so; many pixels in rows that end inside a cache line are the exception: 31 -> 100,
    // 32 x 38 x 38, 12.7 / 11.7 us a float at a time and 13.1 / 13.0 in fours, 16 images 8.4 / 8.6 and 7.2 / 7.8.
    if (hw % 4 == 0 && aligned16(x) && aligned16(y) && (hw % 16 == 0 || g.pixels < 32000)) {
        const int64_t wgs = ceil_div((int64_t)g.pixels, (int64_t)64 * kFewWaves), blocks = ceil_div(cout, 16);
        // four workgroups for each of 256 compute units before a wavefront takes more than one block
        int64_t per = wgs * blocks / 1024;
        per = per < 1 ? 1 : per > kFewVecBlocks ? kFewVecBlocks : per;
        const int64_t parts = ceil_div(blocks, per);
        g.blocks = (int)ceil_div(blocks, parts);
        const dim3 grid((unsigned)wgs, (unsigned)ceil_div(blocks, (int64_t)g.blocks));
#define DML_FEW(KS)                                                                                                       \
    if (cin <= 4 * KS) {                                                                                                  \
        if (w_transposed) hipLaunchKernelGGL((conv_pointwise_few_vec_kernel<KS, true>), grid, 64 * kFewWaves, 0, st, g);  \
        else hipLaunchKernelGGL((conv_pointwise_few_vec_kernel<KS, false>), grid, 64 * kFewWaves, 0, st, g);              \
        return launch_status("conv2d(pointwise, few input channels)");                                                    \
    }
        DML_FEW(4) DML_FEW(6) DML_FEW(8) DML_FEW(10) DML_FEW(12)
#undef DML_FEW
    }
    const int64_t wgs = ceil_div((int64_t)g.pixels, (int64_t)32 * kFewWaves), blocks = ceil_div(cout, 32);
    // two workgroups for each of 256 compute units before a wavefront takes more than one block
    int64_t per = wgs * blocks / 512;
    per = per < 1 ? 1 : per > kFewBlocks ? kFewBlocks : per;
    const int64_t parts = ceil_div(blocks, per);
    g.blocks = (int)ceil_div(blocks, parts);
    const dim3 grid((unsigned)wgs, (unsigned)ceil_div(blocks, (int64_t)g.blocks));
#define DML_FEW(KP)                                                                                                   \
    if (cin <= 2 * KP) {                                                                                              \
        if (w_transposed) hipLaunchKernelGGL((conv_pointwise_few_kernel<KP, true>), grid, 64 * kFewWaves, 0, st, g);  \
        else hipLaunchKernelGGL((conv_pointwise_few_kernel<KP, false>), grid, 64 * kFewWaves, 0, st, g);              \
        return launch_status("conv2d(pointwise, few input channels)");                                                \
    }
    DML_FEW(8) DML_FEW(12) DML_FEW(16) DML_FEW(20) DML_FEW(24)
#undef DML_FEW
    return DMLHIP_ERR_UNSUPPORTED;
}

}  // namespace dml
