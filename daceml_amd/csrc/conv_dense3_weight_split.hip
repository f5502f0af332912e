// Weight gradient of a dense (group 1) 3 x 3 convolution, stride and dilation 1, fp32, on the bf16 matrix instructions: operands
// split into three bf16 values each (bf16_split.h), in the frame of conv_dense3_weight.hip.
//
// Measured, us with the reduction, fp32 instruction and split: 32x64x56x56 -> 64 86 and 71, -> 128 156 and 125, 32x128x28x28 -> 128 86
// and 72, 32x96x40x40 -> 96 125 and 91, 32x256x14x14 -> 256 107 and 104 (rows of 14 are read as 16), 32x64x55x55 -> 64 110 and 99
// (transfers of four bytes). Of the 71 the products are 20, and the split's 80 vector instructions for 18 MFMAs as much beside them; the 48 that
// add the small products take 5, addresses of transfers 9, the ranges' sums and their results 7, the reduction 6.
// The five small products of a tap and sixteen pixels have a sum of their own, which is added to the tap's: 3 roundings of that instead of 12.
// Errors against fp64, 2-norm, fp32 instruction and split (all products in one sum in brackets): 32x64x56x56 -> 64, normal operands, 2.7e-7 and
// 1.3e-7 (2.3e-7), X behind a ReLU 2.1e-7 and 1.3e-7 (2.3e-7), both 5.6e-8 and 2.9e-8 (3.0e-8); 32x128x28x28 -> 256 3.5e-7 and 1.6e-7 (3.2e-7),
// 2.5e-7 and 1.4e-7 (3.0e-7), 4.0e-8 and 3.9e-8 (4.5e-8); 32x256x14x14 -> 256 2.5e-7 and 1.2e-7, 1.8e-7 and 1.1e-7, 4.2e-8 and 4.0e-8. The bf16
// instruction loses the low bits of what it adds in one direction, which 2048 partial sums add up to twice the error: every other
// wavefront adds -dY X instead.
#include "bf16_split.h"
#include "conv_dense3_weight.hip"

namespace dml {
namespace {

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

struct Split {
    static constexpr bool on = true;

    // The products of a chunk: this wavefront's share of its pixels. a_row, x_row: LDS addresses of the lane's rows of dY and X.
    template <int KG, typename Issue>
    static __device__ __forceinline__ void chunk(const WeightArgs& g, floatx16 (&acc)[kTaps], uint32_t a_row, uint32_t x_row, int px, int kg,
                                                 int half, float sign, Issue&& issue_next) {
        // Sixteen pixels at a time: eight next to each other in a row for each lane half, a lane's fragment of dY. The ten
        // values of X they meet in an image row serve three taps: as pairs of bf16 values tap 0 and tap 2 are the same
        // registers one pair apart, tap 1 is shifted by half a register. Reads run one image row ahead and are waited for
        // behind the products they run beside.
        const int g8 = (g.ow + 7) / 8, groups = px / g.ow * g8, steps = (groups + 1) / 2;
        const float inv_g8 = 1.0f / (float)g8;
        uint32_t aa, xa;
        int nv;
        auto locate = [&](int i) {
            const int gi = 2 * i + half, gc = min(gi, groups - 1), r = fast_div(gc, g8, inv_g8), ox = 8 * (gc - r * g8);
            aa = a_row + (uint32_t)((r * g.ow + ox) * 4);
            xa = x_row + (uint32_t)((r * g.pwid + ox + g.col0) * 4);
            nv = gi < groups ? min(8, g.ow - ox) : 0;
        };
        float ra[8], rb[10];
        auto read_a = [&] {
            static_for<0, 8>([&](auto e) { ra[e.value] = lds_read_b32<4 * e.value>(aa); });
        };
        auto read_x = [&](int hy) {
            const uint32_t at = xa + (uint32_t)(hy * g.pwid * 4);
            static_for<0, 10>([&](auto e) { rb[e.value] = lds_read_b32<4 * e.value>(at); });
        };
        auto settle = [&] {
            __builtin_amdgcn_sched_barrier(0);
            wait_lgkm<0>();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 8; ++e) lds_keep(ra[e]);
#pragma unroll
            for (int e = 0; e < 10; ++e) lds_keep(rb[e]);
        };
        if (kg < steps) {
            locate(kg);
            read_a();
            read_x(0);
            settle();
            for (int i = kg; i < steps; i += KG) {
                const int valid = nv;
                const bool partial = __builtin_amdgcn_ballot_w64(valid < 8) != 0;
                if (partial)
#pragma unroll
                    for (int e = 0; e < 8; ++e) ra[e] = e < valid ? ra[e] : 0.f;
                const Pieces pa = split_eight(ra, kSplitScale * sign);
                static_for<0, 3>([&](auto hyc) {
                    constexpr int hy = hyc.value;
                    if (partial)    // what lies behind the row: any bits
#pragma unroll
                        for (int e = 2; e < 10; ++e) rb[e] = e < valid + 2 ? rb[e] : 0.f;
                    uint32_t ph[5], pm[5], pl[5];
#pragma unroll
                    for (int e = 0; e < 5; ++e) split_pair(floatx2{rb[2 * e], rb[2 * e + 1]}, kSplitScale, ph[e], pm[e], pl[e]);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (hy == 2) {
                        locate(min(i + KG, steps - 1));
                        read_a();
                        read_x(0);
                    } else {
                        read_x(hy + 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    // tap 0 and 2 are the same registers, one pair apart; tap 1 lies half a register further on
                    auto fragment = [&](auto tc, const uint32_t (&v)[5]) {
                        constexpr int t = tc.value;
                        u32x4 f;
#pragma unroll
                        for (int e = 0; e < 4; ++e) f[e] = t == 1 ? __builtin_amdgcn_alignbit(v[e + 1], v[e], 16) : v[e + t / 2];
                        return __builtin_bit_cast(bf16x8, f);
                    };
                    static_for<0, 3>([&](auto tc) {
                        constexpr int tap = 3 * hy + tc.value;
                        const Pieces pb = {fragment(tc, ph), fragment(tc, pm), fragment(tc, pl)};
                        acc[tap] = mfma_large(pa, pb, acc[tap]);
                        acc[tap] += mfma_small(pa, pb, floatx16{});
                        asm volatile("" : "+v"(acc[tap]));      // added here, not where the next eights' sums are
                        __builtin_amdgcn_sched_barrier(0);
                    });
                    issue_next();
                    settle();
                });
            }
        }
    }

    // The sums once more where they are not finite. m, c: the lane's rows of dY and X. Returns what gives the sums their size and sign.
    template <int KG, typename ChunkAt>
    static __device__ __forceinline__ float repair(const WeightArgs& g, floatx16 (&acc)[kTaps], ChunkAt&& chunk_at, int first_row, int row_end,
                                                  int m, int c, int kg, int half, float sign) {
        // A value without a split (infinite, NaN, from 2^112 on) makes a sum that is not finite: this wavefront's pixels once more, in fp32
        float bad = 0.f;
#pragma unroll
        for (int t = 0; t < kTaps; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) bad = __builtin_fmaf(acc[t][e], 0.f, bad);
        const bool again = __builtin_amdgcn_ballot_w64(bad != 0.f) != 0;
        if (again) {
#pragma unroll
            for (int t = 0; t < kTaps; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;
            const bool has_m = m < g.m, has_c = c < g.c;
            const int ohw = g.oh * g.ow, in_plane = g.h * g.w;
            const int g8 = (g.ow + 7) / 8;
            auto at = [](bool there, const float* p) { return *(there ? p : reinterpret_cast<const float*>(&g_zeros)); };   // no branches
            for (int r0 = first_row; r0 < row_end;) {
                const Chunk ch = chunk_at(r0);
                const int groups = ch.px / g.ow * g8, steps = (groups + 1) / 2;
                for (int i = kg; i < steps; i += KG) {
                    const int gi = 2 * i + half, r = gi / g8, ox0 = 8 * (gi - r * g8);
                    const int oy = ch.oy + r;
                    float av[8], xv[3][10];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        av[e] = at(gi < groups && ox0 + e < g.ow && has_m, g.dy + ((int64_t)ch.img * g.m + m) * ohw + oy * g.ow + ox0 + e) * sign;
#pragma unroll
                    for (int hy = 0; hy < 3; ++hy)
#pragma unroll
                        for (int e = 0; e < 10; ++e) {
                            const int iy = oy - g.ph + hy, ix = ox0 - g.pw + e;
                            const bool in = gi < groups && ox0 + e < g.ow + 2 && has_c && iy >= 0 && iy < g.h && ix >= 0 && ix < g.w;
                            xv[hy][e] = at(in, g.x + ((int64_t)ch.img * g.c + c) * in_plane + iy * g.w + ix);
                        }
#pragma unroll
                    for (int e = 0; e < 8; ++e)
#pragma unroll
                        for (int t = 0; t < kTaps; ++t) {
                            const float bv = ox0 + e < g.ow ? xv[t / 3][e + t % 3] : 0.f;
                            acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[e], bv, acc[t], 0, 0, 0);
                        }
                }
                r0 += ch.px / g.ow;
            }
        }
        return again ? sign : sign * kSplitBack;
    }
};

template <int WM, int AVEC, int XVEC>
__global__ __launch_bounds__(kThreads) void conv_dense3_weight_split_kernel(const WeightArgs g) {
    weight_gradient<WM, AVEC, XVEC, Split>(g);
}

}  // namespace

int launch_conv_dense3_weight(const ConvGeom& g, const float* x, const float* dy, float* part, hipStream_t st) {
    constexpr size_t kReadPast = 64;      // the last pixels of a row are read in eights, past the end of what is staged
    WeightPlan pl;
    unsigned blocks;
    int avec, xvec;
    // Rows are read as whole eights of pixels: not where that is more than 1.42 times as many. Times those of the fp32 instruction, 5 - 65 columns,
    // 64 - 192 channels: 5, 6, 9, 10, 11 columns 1.18 - 1.29, 1.07 - 1.18, 0.97 - 1.08, 0.98 - 1.03, 0.98 - 1.03; 7 columns 0.94 - 1.07; 8 and
    // 12 - 65 0.73 - 1.01 (17 to 19 columns 0.97 - 1.01, whole eights 0.73 - 1.00).
    const bool eights = g.ow >= 8 && 100 * ceil_div(g.ow, 8) * 8 <= 142 * g.ow;
    const bool split = eights && g.sh == 1 && g.sw == 1 && g.dh == 1 && g.dw == 1 && plan_weight(g, x, dy, &pl, &blocks, &avec, &xvec) &&
                       pl.lds + kReadPast <= (size_t)kLdsBytes;
    if (!split) return launch_conv_dense3_bwd_weight(g, x, dy, part, st);
    pl.lds += kReadPast;
    note_conv_form(20);
    pl.a.x = x; pl.a.dy = dy; pl.a.part = part;
    const int wm = g.m > 32 ? 2 : 1;
#define DML_D3W(WM, AV, XV) \
    if (wm == WM && avec == AV && xvec == XV) return launch_weight(conv_dense3_weight_split_kernel<WM, AV, XV>, pl, blocks, st);
    DML_D3W(1, 1, 1) DML_D3W(1, 1, 4) DML_D3W(1, 4, 1) DML_D3W(1, 4, 4)
    DML_D3W(2, 1, 1) DML_D3W(2, 1, 4) DML_D3W(2, 4, 1) DML_D3W(2, 4, 4)
#undef DML_D3W
    return DMLHIP_ERR_UNSUPPORTED;
}

}  // namespace dml
