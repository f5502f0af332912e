// 1x1 convolutions of many input and few output channels, fp32 (the projection of an inverted-residual block, with or without
// the squeeze-excite gate on its input, and the data gradient of its expansion):
//   Y[n, m, p] = act(sum_c W[m, c] (s[n, c] X[n, c, p]) + b[m])
//
// What bounds them: reading X once, the matrix pipe is at half of that. A wavefront takes up to 64 pixels and all output channels on
// v_mfma_f32_16x16x4_f32: lane q of a group of sixteen has four consecutive pixels, group k input channel 4 s + k, so X is read in
// pieces of 256 bytes (16 bytes per lane) straight into the registers the product takes it from, 16 - 48 input channels ahead of the
// product, and Y leaves in pieces of 256 bytes. Blocks of 16 output channels waste less on 24, 40 or 48 of them than blocks of 32.
// Only the weights are in LDS, some hundred input channels at a time. Measured, us, the kernels before and here: 192 -> 48
// channels, 96 x 56 x 56, gated 107 and 70 (289 MB, 4.1 TB/s), 144 -> 24, 32 x 56 x 56, 36 and 22, data gradient 24 and 21.
#include "common.h"
#include "conv_geom.h"

#include <type_traits>

namespace dml {
namespace {

constexpr int kProjThreads = 256;
constexpr int kProjMaxOut = 80;              // output channels: 5 blocks of 16
constexpr int kProjGroup = 16;               // input channels that are loaded together
constexpr int kProjLds = 40 * 1024;          // weights of a chunk: three workgroups per compute unit
constexpr uint32_t kProjNothing = 0x80000000u;   // buffer offset past the end of every buffer: loads return zero
constexpr int kProjBufferFlags = 0x00020000; // raw buffer of 32-bit data

struct ProjArgs {
    const float* x;
    const float* w;
    const float* bias;
    const float* gate;
    float* y;
    int n, cin, cout, act, transposed, wvec; // transposed: w is [cin][cout]; wvec: [cout][cin] in whole vectors
    uint32_t hw, pixels;                     // of an image, of all
    int chunk;                               // groups of input channels whose weights are in LDS, a multiple of four
};

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// MT: blocks of 16 output channels. PB: blocks of 16 pixels per wavefront. VEC: consecutive pixels per lane, PB or 1.
template <int MT, int PB, int VEC>
__global__ __launch_bounds__(kProjThreads, MT == 5 ? 2 : 3) void conv_pointwise_project_kernel(const ProjArgs g) {
    constexpr int NV = PB / VEC, RING = PB == 4 ? 2 : 4;   // groups of input channels in registers
    constexpr int kPitch = 16 * (MT | 1);    // rows of four input channels start in different quarters of the banks
    extern __shared__ float ws[];
    const int lane = threadIdx.x & 63, q = lane & 15, kk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t p0 = (blockIdx.x * 4u + (uint32_t)wave) * (16u * PB) + (uint32_t)(VEC * q);

    const auto xbuf = __builtin_amdgcn_make_buffer_rsrc((void*)g.x, 0, (int)((uint32_t)g.cin * g.pixels * 4u), kProjBufferFlags);
    const auto gbuf = __builtin_amdgcn_make_buffer_rsrc((void*)g.gate, 0, g.n * g.cin * 4, kProjBufferFlags);
    const bool gated = g.gate != nullptr;
    uint32_t xoff[NV], goff[NV], yoff[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const uint32_t p = p0 + 16u * v;
        const bool ok = p < g.pixels;
        const uint32_t img = ok ? p / g.hw : 0u, r = p - img * g.hw;
        xoff[v] = ok ? ((img * (uint32_t)g.cin + kk) * g.hw + r) * 4u : kProjNothing;
        goff[v] = ok ? (img * (uint32_t)g.cin + kk) * 4u : kProjNothing;
        yoff[v] = ok ? img * (uint32_t)g.cout * g.hw + r : kProjNothing;
    }
    float xr[RING][4][PB], gr[RING][4][NV];
    const int groups = (g.cin + kProjGroup - 1) / kProjGroup;
    auto issue = [&](auto slotc, int group) {
        constexpr int SLOT = decltype(slotc)::value;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int c = group * kProjGroup + 4 * s;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                // an input channel past the last one lies in the next image
                const uint32_t off = c + kk < g.cin ? xoff[v] : kProjNothing;
                if constexpr (VEC == 4) {
                    const floatx4 u = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(xbuf, off, c * (int)g.hw * 4, 0));
#pragma unroll
                    for (int e = 0; e < 4; ++e) xr[SLOT][s][e] = u[e];
                } else {
                    xr[SLOT][s][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, off, c * (int)g.hw * 4, 0));
                }
                if (gated)
                    gr[SLOT][s][v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                                   gbuf, c + kk < g.cin ? goff[v] : kProjNothing, c * 4, 0));
            }
        }
    };
    floatx4 acc[MT][PB];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < PB; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // Weights of the groups from `first` on, zero past the last input and output channel. Rows of whole vectors are read sixteen
    // bytes at a time, the others a float at a time, eight loads before the first store.
    auto stage = [&](int first) {
        const int c0 = first * kProjGroup, count = min(g.chunk, groups - first);
        if (g.wvec) {
            for (int t0 = wave; t0 < count * MT; t0 += 4 * 4) {
                floatx4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int t = min(t0 + 4 * u, count * MT - 1), k = t / MT, m = (t - k * MT) * 16 + q, c = c0 + 16 * k + 4 * kk;
                    const bool in = c < g.cin && m < g.cout;
                    v[u] = *reinterpret_cast<const floatx4*>(g.w + (in ? (size_t)m * g.cin + c : 0));
                    v[u] = in ? v[u] : floatx4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int t = min(t0 + 4 * u, count * MT - 1), k = t / MT;
#pragma unroll
                    for (int e = 0; e < 4; ++e) ws[(16 * k + 4 * kk + e) * kPitch + (t - k * MT) * 16 + q] = v[u][e];
                }
            }
            return;
        }
        const int steps = count * (kProjGroup / 4);
        for (int t0 = wave; t0 < steps * MT; t0 += 4 * 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int t = min(t0 + 4 * u, steps * MT - 1), s = t / MT, m = (t - s * MT) * 16 + q, c = c0 + 4 * s + kk;
                const bool in = c < g.cin && m < g.cout;
                const float wv = g.w[!in ? 0 : g.transposed ? (size_t)c * g.cout + m : (size_t)m * g.cin + c];
                v[u] = in ? wv : 0.f;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int t = min(t0 + 4 * u, steps * MT - 1), s = t / MT;
                ws[(4 * s + kk) * kPitch + (t - s * MT) * 16 + q] = v[u];
            }
        }
    };
    auto multiply = [&](auto slotc, const float* wg) {
        constexpr int SLOT = decltype(slotc)::value;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            float a[MT], b[PB];
#pragma unroll
            for (int i = 0; i < MT; ++i) a[i] = wg[(4 * s + kk) * kPitch + i * 16 + q];
#pragma unroll
            for (int j = 0; j < PB; ++j) b[j] = gated ? xr[SLOT][s][j] * gr[SLOT][s][VEC == 1 ? j : 0] : xr[SLOT][s][j];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < PB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };

    static_for<0, RING>([&](auto r) {
        if (r.value < groups) issue(r, r.value);
    });
    for (int first = 0; first < groups; first += g.chunk) {
        __syncthreads();                     // the weights before these have been multiplied
        stage(first);
        __syncthreads();
        const int end = min(first + g.chunk, groups);
        for (int k0 = first; k0 < end; k0 += RING)
            static_for<0, RING>([&](auto r) {
                const int k = k0 + r.value;
                if (k >= end) return;
                multiply(r, ws + (k - first) * kProjGroup * kPitch);
                if (k + RING < groups) issue(r, k + RING);
            });
    }

    // element e of a block: output channel 4 kk + e of its sixteen, the pixel of lane q
    auto all = [&](auto actc) {
        constexpr int ACT = decltype(actc)::value;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int m = i * 16 + 4 * kk + e;
                if (m >= g.cout) continue;
                const float b = g.bias ? g.bias[m] : 0.f;
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    if (yoff[v] == kProjNothing) continue;
                    float* const o = g.y + yoff[v] + (size_t)m * g.hw;
                    if constexpr (VEC == 4)
                        *reinterpret_cast<floatx4*>(o) =
                            floatx4{apply_act(ACT, acc[i][0][e] + b), apply_act(ACT, acc[i][1][e] + b),
                                    apply_act(ACT, acc[i][2][e] + b), apply_act(ACT, acc[i][3][e] + b)};
                    else
                        *o = apply_act(ACT, acc[i][v][e] + b);
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

template <int MT>
int launch_project(ProjArgs& g, bool vec, hipStream_t st) {
    const int pitch = 16 * (MT | 1), groups = (g.cin + kProjGroup - 1) / kProjGroup;
    g.chunk = kProjLds / (kProjGroup * pitch * 4) & ~3;
    if (g.chunk > groups) g.chunk = (groups + 3) & ~3;
    const size_t lds = (size_t)g.chunk * kProjGroup * pitch * sizeof(float);
    // Pixels per wavefront, us with 16 / 32 / 64: 12 images of 56 x 56, 192 -> 48 channels, 19.7 / 20.7 / 19.7, 96 images 100 / 78 / 67;
    // pixels that are not read in fours take a load each, 12 images of 55 x 55, 144 -> 40, 15.8 / 18.1 / 22.6, 32 images 29 / 26 / 30.
    const int pb = vec ? (g.pixels >= 40000 ? 4 : 1) : g.pixels >= 60000 ? 2 : 1;
    const unsigned grid = (unsigned)ceil_div((int64_t)g.pixels, (int64_t)4 * 16 * pb);
    const auto kern = pb == 1 ? conv_pointwise_project_kernel<MT, 1, 1>
                      : vec ? conv_pointwise_project_kernel<MT, 4, 4> : conv_pointwise_project_kernel<MT, 2, 1>;
    hipLaunchKernelGGL(kern, grid, kProjThreads, lds, st, g);
    return launch_status("conv2d(pointwise, few output channels)");
}

}  // namespace

// streams: the other choice is the kernel of conv.hip that takes X through LDS, slower everywhere (192 -> 48 channels, 12 / 32 / 96 images of
// 56 x 56, 24 / 40 / 91 us and 20 / 30 / 67; with the gate 27 / 42 / 107 and 20 / 30 / 70; 480 -> 80, one image of 14 x 14, 62 and 30). The tiled
// GEMM spreads few pixels over more wavefronts: forward, 12 / 32 / 96 images of 55 x 55, 144 -> 40, 19 / 35 / 92 and 16 / 26 / 63, one
// image 5.6 and 9.4; 240 -> 40, 32 / 96 images of 27 x 27, 19.5 / 41 and 18 / 35; transposed weights are read a float at a time: 12 / 32 / 96
// images of 55 x 55 16 / 29 / 74 and 18 / 28 / 66, 240 -> 40, 96 images of 27 x 27, 34 and 38.
bool pointwise_project_applicable(int64_t n, int64_t cin, int64_t cout, int64_t hw, bool w_transposed, bool streams) {
    if (cin < 64 || cin < 2 * cout || cout < 1 || cout > kProjMaxOut || hw < 32 || n * hw * cin >= (1LL << 29)) return false;
    if (streams) return true;
    return w_transposed ? cin <= 160 && n * hw >= 90000 : n * hw >= (cin <= 160 ? 30000 : 60000);
}

// With few pixels a wavefront's chain over all input channels is what takes the time; the tiled GEMM cuts it into pieces. us, here and
// there: 480 -> 80, one image of 14 x 14, 30 and 6, 96 images 42 and 27; 240 -> 40, 1 / 20 / 48 images of 28 x 28, 16 / 17 / 25 and 5 / 12 / 24; 144 -> 24, 3 / 9
// images of 56 x 56, 8.9 / 10.7 and 6.5 / 13.0; 96 -> 16, one image of 112 x 112, 5.0 and 5.7.
bool pointwise_splits_channels(int64_t n, int64_t cin, int64_t cout, int64_t hw) {
    return cin >= 96 && cin >= 2 * cout && cout <= kProjMaxOut && n * hw < 64 * cin;
}

int launch_pointwise_project(const float* x, const float* w, const float* bias, const float* gate, float* y, int n, int cin,
                             int cout, int64_t hw, int act, bool w_transposed, hipStream_t st) {
    ProjArgs g;
    g.x = x; g.w = w; g.bias = bias; g.gate = gate; g.y = y;
    g.n = n; g.cin = cin; g.cout = cout; g.act = act; g.transposed = w_transposed;
    g.hw = (uint32_t)hw;
    g.pixels = (uint32_t)(n * hw);
    g.wvec = !w_transposed && cin % 4 == 0 && aligned16(w);
    const bool vec = hw % 4 == 0 && aligned16(x) && aligned16(y);
    switch ((cout + 15) / 16) {
        case 1: return launch_project<1>(g, vec, st);
        case 2: return launch_project<2>(g, vec, st);
        case 3: return launch_project<3>(g, vec, st);
        case 4: return launch_project<4>(g, vec, st);
        default: return launch_project<5>(g, vec, st);
    }
}

}  // namespace dml
