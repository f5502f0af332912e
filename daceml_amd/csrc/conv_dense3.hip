// Dense (group 1) 3 x 3 convolution, fp32, as an implicit GEMM on v_mfma_f32_32x32x2_f32 that streams its operands
// straight into LDS; the forward pass and, with the weights read transposed and reversed, the data gradient. For problems of fewer
// tiles or channels than conv_dense3_split.hip takes, which is asked first.
//   Y[n, m, p] = act(b[m] + sum_{c, hy, hx} W[m, c, hy, hx] * X[n, c, oy(p) s - pad + hy d, ox(p) s - pad + hx d])
//
// What bounds it: the fp32 matrix rate (256 operations per clock and compute unit), if the matrix pipes neither wait for
// operands nor for the last of too few workgroups. So
// - a wavefront computes one 32 x 32 block, and a tile's pixels are counted through the whole batch, not per image: 32 images
//   of 56 x 56 in 64 channels are 6.1 workgroups of 32 x 128 per compute unit (tiles of 64 x 256 per image were 1.6, a
//   fifth of the chip idle). Where even that is too few, wavefronts split the input channels of a 32 x 64 or 32 x 32 tile;
// - a step is 4 input channels (x the wavefronts that split them). The rectangle of X under the tile's pixels and the step's
//   weights go global -> LDS without staging registers, one step ahead, between the MFMAs of the step before; every
//   tap is a shifted read of the same rectangle. One barrier per step; small steps leave room for four workgroups on a
//   compute unit, whose first loads and stores then hide behind each other's products. Rows of X whose length is a multiple
//   of four floats move 16 bytes per lane (4 bytes per lane: 106 us where 16 take 88).
// Measured, us forward / data gradient, before (general implicit-GEMM kernel) and now: 32x64x56x56 -> 64 118 / 120 and
// 88 / 87, 32x256x14x14 -> 256 362 / 341 and 107 / 106, 1x256x14x14 -> 256 353 / 334 and 41 / 42; at the matrix rate that a
// large product reaches the first two take 48. The rest: 6.1 workgroups per compute unit are seven for some (62 us at a
// product's pace), first loads and stores 12 us, operand transfers 13 us (timed with the later steps' transfers left out).
// A = W (rows = output channels), B = X (columns = pixels). The two lane halves of an MFMA multiply different channels of the
// step. Steps of 8 channels, tiles of 64 x 64 and 64 x 128 measured 94 - 108 us for the first problem.
#include "common.h"
#include "conv_geom.h"
#include "lds_ops.h"

#include <type_traits>

namespace dml {
namespace {

constexpr int kTaps = 9;
constexpr int kMaxPieces = 4;     // 256-float pieces of a channel's rectangle
constexpr int kHalf = 2;          // channels per lane half of an MFMA and step
constexpr int kCus = 256;
constexpr int64_t kMaxBlocks = (1 << 24) - 1;   // of 256 threads: a grid has less than 2^32 threads

__device__ const floatx4 g_zeros = {0.f, 0.f, 0.f, 0.f};   // what lanes outside an operand read

struct Dense3Args {
    const float* x;
    const float* w;
    const float* bias;
    float* y;
    int n, c, h, w_in, m, sh, sw, ph, pw, dh, dw, oh, ow, act;
    int img_rows;             // rows of a padded image: rectangles are cut from the images stacked on each other
    int pwid, rect, plane;    // rectangle columns, floats, and pitch per channel in LDS (the planes of the lane halves differ
                              // by half the banks)
    int x_bytes;              // all of a step's rectangles in LDS
    int col0;                 // rectangle column of the padded image's column 0
    int ids_h, ids_w;         // data gradient: dY is read as if ids - 1 zeros stood between its rows / columns
    int total_px, tiles_m;
};

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

template <int BYTES>
__device__ __forceinline__ void lds_dma(const float* gptr, char* lds_dst) {
    const auto g = (const __attribute__((address_space(1))) void*)gptr;
    const auto l = (__attribute__((address_space(3))) void*)lds_dst;
    if constexpr (BYTES == 16) __builtin_amdgcn_global_load_lds(g, l, 16, 0, 0);
    else __builtin_amdgcn_global_load_lds(g, l, 4, 0, 0);
}

// Offset of the filter of a (channel, channel) pair. The product and the sum that follows are kept apart: as one 64-bit
// multiply-add the sum's operand has a high half that nothing wrote, and the register it names may belong to an LDS read in
// flight - harmless, its result is cut off, but the same to see as the hazard that lds_ops.h describes.
__device__ __forceinline__ uint32_t taps_of(uint32_t pair) {
    uint32_t at = pair * kTaps;
    asm volatile("" : "+v"(at));
    return at;
}

// The weights of a step in LDS. Forward: rows of one output channel, 9 CH floats and 4 of padding (16 rows 12 or 36 banks
// apart start in 16 different groups of four banks). FLIP: as they lie in memory for one input channel, [CH][MB][9].
template <int MB, int CH, bool FLIP, int VEC>
struct Weights {
    static constexpr int PITCH = CH * kTaps + (CH == 4 ? 8 : 4);   // an odd multiple of four banks
    static constexpr int FLOATS = FLIP ? CH * MB * kTaps : MB * PITCH;
    static constexpr int INSTR = (FLOATS + 64 * VEC - 1) / (64 * VEC);      // transfers of a step
    static constexpr int BYTES = INSTR * 64 * VEC * 4;                      // all of them, padding included
    static constexpr int PER_WAVE = (INSTR + 3) / 4;
    // transfer i of wavefront `wave`; c0: first input channel of the step
    static __device__ __forceinline__ void issue(const Dense3Args& g, int i, int wave, int lane, int m0, int c0, char* dst) {
        if (i * 4 + wave >= INSTR) return;
        const int f = ((i * 4 + wave) * 64 + lane) * VEC;
        const float* src;
        bool ok;
        if constexpr (FLIP) {      // W is [input channel of this product][output channel][9]
            const int ch = f / (MB * kTaps), j = f % (MB * kTaps);
            ok = f < FLOATS && c0 + ch < g.c && j < (g.m - m0) * kTaps;
            src = g.w + (taps_of((uint32_t)((c0 + ch) * g.m + m0)) + (uint32_t)j);
        } else {
            const int row = f / PITCH, k = f % PITCH;
            ok = row < MB && m0 + row < g.m && k < min(CH, g.c - c0) * kTaps;
            src = g.w + (taps_of((uint32_t)((m0 + row) * g.c + c0)) + (uint32_t)k);
        }
        if (!ok) src = reinterpret_cast<const float*>(&g_zeros);
        lds_dma<VEC * 4>(src, dst + (i * 4 + wave) * 64 * VEC * 4);
    }
};

// Tile: 32 output channels x 32 WP pixels, one 32 x 32 block per wavefront; KG wavefronts split the input channels of a
// block's step. VEC, XVEC: floats per lane and transfer of the weights and of X.
template <int WP, int KG, bool FLIP, int VEC, int XVEC>
__global__ __launch_bounds__(256) void conv_dense3_f32_kernel(const Dense3Args g) {
    static_assert(WP * KG == 4, "four wavefronts");
    constexpr int MB = 32, PX = 32 * WP, CH = 2 * kHalf * KG;
    typedef Weights<MB, CH, FLIP, VEC> W;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int stage_bytes = g.x_bytes + W::BYTES;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int l32 = lane & 31, half = lane >> 5;
    const int kg = wave / WP, wp = wave % WP;
    const int ch0 = (kg * 2 + half) * kHalf;             // this lane half's first channel of a step
    // the tiles of one stretch of pixels follow each other: they read the same X
    const int m0 = (int)(blockIdx.x % (unsigned)g.tiles_m) * MB;
    const int p0 = (int)(blockIdx.x / (unsigned)g.tiles_m) * PX;
    const int ohw = g.oh * g.ow;
    const float inv_ohw = 1.0f / (float)ohw, inv_ow = 1.0f / (float)g.ow, inv_rows = 1.0f / (float)g.img_rows;

    // pixel p of the batch reads row n img_rows + oy sh + hy dh of the stacked images, column ox sw + hx dw
    const int n_first = p0 / ohw, q_first = p0 - n_first * ohw;
    const int r_first = q_first / g.ow * g.sh;        // in its image
    const int row_first = n_first * g.img_rows + r_first;
    const uint32_t lds0 = lds_addr(lds);
    const int p = p0 + wp * 32 + l32;                 // this lane's column
    uint32_t xaddr;
    {
        const int q0 = min(p, g.total_px - 1) - p0 + q_first;
        const int n = fast_div(q0, ohw, inv_ohw), q = q0 - n * ohw;
        const int oy = fast_div(q, g.ow, inv_ow), ox = q - oy * g.ow;
        xaddr = lds0 + (uint32_t)(((n * g.img_rows + oy * g.sh - r_first) * g.pwid + ox * g.sw + g.col0 + ch0 * g.plane) * 4);
    }
    const uint32_t waddr = lds0 + (uint32_t)g.x_bytes +
                           (uint32_t)((FLIP ? (ch0 * MB + l32) * kTaps : l32 * W::PITCH + ch0 * kTaps) * 4);

    // What this lane transfers. 4 bytes at a time: up to four positions of every channel's rectangle, whose rows start with
    // the left padding. 16 bytes: pieces of the whole step's rectangles; the rows hold whole rows of X, between them
    // four zeros that pad the one on its right and the other on its left.
    constexpr int NX = kMaxPieces * (XVEC == 4 && KG == 4 ? 2 : 1);
    const float* src[NX];
    int64_t next[NX];                    // to the next channel / step
    int chan[NX];
    const int in_plane = g.h * g.w_in;
#pragma unroll
    for (int u = 0; u < NX; ++u) {
        int pos = (u * 4 + wave) * 64 + lane;
        int row, iy, ix;
        chan[u] = 0;
        bool ok;
        if constexpr (XVEC == 4) {
            chan[u] = fast_div(pos * 4, g.plane, 1.0f / (float)g.plane);
            pos = pos * 4 - chan[u] * g.plane;
            row = fast_div(max(pos - 4, 0), g.pwid, 1.0f / (float)g.pwid);
            ix = pos - 4 - row * g.pwid;
            ok = pos >= 4 && pos < g.rect && chan[u] < CH;
        } else {
            row = fast_div(pos, g.pwid, 1.0f / (float)g.pwid);
            ix = pos - row * g.pwid - g.pw;
            ok = pos < g.rect;
        }
        const int n = fast_div(r_first + row, g.img_rows, inv_rows);
        iy = r_first + row - n * g.img_rows - g.ph;
        ok = ok && n_first + n < g.n && iy >= 0 && ix >= 0;
        if (XVEC == 1 && (g.ids_h > 1 || g.ids_w > 1)) {
            const int qy = max(iy, 0) / g.ids_h, qx = max(ix, 0) / g.ids_w;
            ok = ok && qy * g.ids_h == iy && qx * g.ids_w == ix;
            iy = qy;
            ix = qx;
        }
        ok = ok && iy < g.h && ix < g.w_in;
        src[u] = ok ? g.x + (((int64_t)(n_first + n) * g.c + chan[u]) * in_plane + (iy * g.w_in + ix))
                    : reinterpret_cast<const float*>(&g_zeros);
        next[u] = ok ? (int64_t)in_plane * (XVEC == 4 ? CH : 1) : 0;
    }
    // part `part` of CH / 2 of the step that starts at channel c0
    auto issue_x = [&](auto part_c, int c0, char* stage) {
        constexpr int part = decltype(part_c)::value, PARTS = CH / 2;
        if constexpr (XVEC == 4) {
#pragma unroll
            for (int u = part * NX / PARTS; u < (part + 1) * NX / PARTS; ++u) {
                if ((u * 4 + wave) * 256 >= CH * g.plane) continue;
                lds_dma<16>(c0 + chan[u] < g.c ? src[u] : reinterpret_cast<const float*>(&g_zeros), stage + (u * 4 + wave) * 1024);
                src[u] += next[u];
            }
        } else {
#pragma unroll
            for (int ch = part * 2; ch < part * 2 + 2; ++ch) {
                const bool in = c0 + ch < g.c;
#pragma unroll
                for (int u = 0; u < NX; ++u) {
                    if ((u * 4 + wave) * 64 >= g.rect) continue;
                    lds_dma<4>(in ? src[u] : reinterpret_cast<const float*>(&g_zeros), stage + (ch * g.plane + (u * 4 + wave) * 64) * 4);
                    if (in) src[u] += next[u];
                }
            }
        }
    };
    auto issue_w = [&](int i, int c0, char* stage) { W::issue(g, i, wave, lane, m0, c0, stage + g.x_bytes); };

    floatx16 acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.f;

    // two fragments of the 18 (channel, tap) pairs of this lane half: pair f is channel f / 9, tap f % 9
    float af[2][kHalf], bf[2][kHalf];
    auto frags = [&](auto qc, uint32_t so, float (&a)[kHalf], float (&b)[kHalf]) {
        constexpr int q = decltype(qc)::value;
        static_for<0, kHalf>([&](auto ec) {
            constexpr int e = decltype(ec)::value, f = q * kHalf + e, t = f % kTaps;
            a[e] = lds_read_b32<(FLIP ? f / kTaps * MB * kTaps + kTaps - 1 - t : f) * 4>(waddr + so);
            b[e] = lds_read_b32<0>(xaddr + so + (uint32_t)((f / kTaps * g.plane + t / 3 * g.dh * g.pwid + t % 3 * g.dw) * 4));
        });
    };

    const int steps = (g.c + CH - 1) / CH;
    static_for<0, CH / 2>([&](auto pc) { issue_x(pc, 0, lds); });
#pragma unroll
    for (int i = 0; i < W::PER_WAVE; ++i) issue_w(i, 0, lds);
    wait_vm_lgkm0<0>();
    __builtin_amdgcn_s_barrier();
    frags(std::integral_constant<int, 0>{}, 0u, af[0], bf[0]);

    int t = 0;
    auto step = [&](auto more_c) {
        constexpr bool MORE = decltype(more_c)::value;
        const uint32_t so = (uint32_t)((t & 1) * stage_bytes), sn = (uint32_t)stage_bytes - so;
        char* const nxt = lds + sn;
        static_for<0, kTaps>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            // the fragments alternate between two register sets; nine per step, so odd steps start with the other one:
            // they are copied over at the end of the step instead
            constexpr int cur = q & 1, nb = (q + 1) & 1;
            wait_lgkm<0>();
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, kHalf>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(af[cur][e], bf[cur][e], acc, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (e == 0 && q < kTaps - 1) {
                    frags(std::integral_constant<int, q + 1>{}, so, af[nb], bf[nb]);
                } else if constexpr (e == 0 && MORE) {
                    // every fragment of this step is in registers and the next step has landed, for all wavefronts
                    // behind the barrier: this stage is free
                    wait_vm_lgkm0<0>();
                    __builtin_amdgcn_s_barrier();
                    frags(std::integral_constant<int, 0>{}, sn, af[nb], bf[nb]);
                }
                if constexpr (MORE && e == 1 && q < 5) {
                    if constexpr (q < 4)
                        static_for<q * (CH / 2) / 4, (q + 1) * (CH / 2) / 4>([&](auto pc) { issue_x(pc, (t + 1) * CH, nxt); });
                    constexpr int i0 = q * W::PER_WAVE / 5, i1 = (q + 1) * W::PER_WAVE / 5;
#pragma unroll
                    for (int i = i0; i < i1; ++i) issue_w(i, (t + 1) * CH, nxt);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        if constexpr (MORE) {
            wait_lgkm<0>();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < kHalf; ++e) {
                af[0][e] = af[1][e];
                bf[0][e] = bf[1][e];
            }
        }
        ++t;
    };
    while (t + 1 < steps) step(std::true_type{});
    step(std::false_type{});

    // element e of a block: row (e / 4) * 8 + (lane / 32) * 4 + e % 4, column lane % 32
    if constexpr (KG > 1) {
        constexpr int PITCH = PX + 1;
        __syncthreads();                 // the stages are done with
        float* part = reinterpret_cast<float*>(lds);
#pragma unroll
        for (int e = 0; e < 16; ++e) part[(kg * 32 + (e >> 2) * 8 + half * 4 + (e & 3)) * PITCH + wp * 32 + l32] = acc[e];
        __syncthreads();
        const int px = (int)threadIdx.x % PX, po = p0 + px;
        if (po >= g.total_px) return;
        const int n = po / ohw, q = po - n * ohw;
#pragma unroll
        for (int r = 0; r < 32 * PX / 256; ++r) {
            const int row = r * (256 / PX) + (int)threadIdx.x / PX, m = m0 + row;
            if (m >= g.m) continue;
            const float* s = part + row * PITCH + px;
            float v = s[0] + s[32 * PITCH];
            if constexpr (KG == 4) v += s[64 * PITCH] + s[96 * PITCH];
            g.y[((int64_t)n * g.m + m) * ohw + q] = apply_act(g.act, v + (g.bias ? g.bias[m] : 0.f));
        }
    } else {
        if (p >= g.total_px) return;
        const int mw = m0 + half * 4;
        const int n = p / ohw, q = p - n * ohw;
        float* out = g.y + (int64_t)n * g.m * ohw + q;
        float b[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = mw + (e >> 2) * 8 + (e & 3);
            b[e] = g.bias && m < g.m ? g.bias[m] : 0.f;
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = mw + (e >> 2) * 8 + (e & 3);
            if (m < g.m) out[(int64_t)m * ohw] = apply_act(g.act, acc[e] + b[e]);
        }
    }
}

// Tile t: 128 >> t pixels, 1 << t wavefronts that split the input channels, 4 << t of them per step. The one with the least
// estimated time is taken: a step of a workgroup that has its compute unit to itself, and of one among several, in us as
// measured, and 3 us for first loads and stores per round of resident workgroups. X that moves 4 bytes per lane adds to a step
// for every transfer: its instructions, and LDS that leaves no room for another workgroup. What it decides (n x c x size -> m,
// us for the three tiles): 32x64x56->64 87 / 87 / 130, 12x128x28->128 51 / 40 / 46, 1x256x14->256 77 / 52 / 41; of odd sizes
// 32x32x114->64 211 / 345 / 938, 12x128x29->128 62 / 50 / 76, 4x128x29->128 47 / 32 / 31.
constexpr int kTiles = 3;
constexpr double kStepAlone[kTiles] = {1.15, 1.5, 2.2}, kStepShared[kTiles] = {0.76, 0.8, 1.05};
constexpr double kNarrowTransfer[kTiles] = {0.004, 0.004, 0.008};

struct Dense3Plan {
    Dense3Args a;
    double us;               // estimated
    int tile, vec, xvec;
    size_t lds;
    unsigned blocks;
};

thread_local int g_force_tile = -1;

size_t weight_bytes(int tile, bool flip, int vec) {
#define DML_WB(T)                                                                                                      \
    if (tile == T)                                                                                                     \
        return flip ? (vec == 4 ? Weights<32, 2 * kHalf << T, true, 4>::BYTES : Weights<32, 2 * kHalf << T, true, 1>::BYTES) \
                    : (vec == 4 ? Weights<32, 2 * kHalf << T, false, 4>::BYTES : Weights<32, 2 * kHalf << T, false, 1>::BYTES);
    DML_WB(0) DML_WB(1) DML_WB(2)
#undef DML_WB
    return 0;
}

template <int TILE, bool FLIP, int VEC, int XVEC>
int launch_tile(const Dense3Plan& pl, hipStream_t st, const char* what) {
    auto kern = conv_dense3_f32_kernel<(4 >> TILE), (1 << TILE), FLIP, VEC, XVEC>;
    if (pl.lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds);
        if (e != hipSuccess) {
            set_error("%s: cannot reserve %zu bytes of LDS: %s", what, pl.lds, hipGetErrorString(e));
            return (int)e;
        }
    }
    hipLaunchKernelGGL(kern, pl.blocks, 256, pl.lds, st, pl.a);
    return launch_status(what);
}

template <bool FLIP, int VEC, int XVEC>
int launch_form(const Dense3Plan& pl, hipStream_t st, const char* what) {
    if (pl.tile == 0) return launch_tile<0, FLIP, VEC, XVEC>(pl, st, what);
    if (pl.tile == 1) return launch_tile<1, FLIP, VEC, XVEC>(pl, st, what);
    return launch_tile<2, FLIP, VEC, XVEC>(pl, st, what);
}

}  // namespace

// The geometry is the product's own: for a data gradient the stride-1 convolution of the (zero-dilated) dY. False where a
// tile's rectangle is too large for LDS, an extent for 32-bit arithmetic or the grid, or where the general kernel applies
// (`general`) and is the faster one.
static bool plan_conv_dense3(const ConvGeom& g, int ids_h, int ids_w, bool flip, bool general, const void* x, const void* w,
                             Dense3Plan* pl) {
    if (g.kh != 3 || g.kw != 3 || g.group != 1 || g.n < 1 || g.c < 4 || g.m < 1 || g.oh < 1 || g.ow < 1) return false;
    const int64_t ohw = (int64_t)g.oh * g.ow, total = (int64_t)g.n * ohw;
    if ((double)total * g.m * g.c * kTaps < (double)(1 << 24)) return false;     // tiny: the direct kernel
    const int64_t img_rows = (int64_t)(g.oh - 1) * g.sh + 2LL * g.dh + 1;
    const int64_t pwid = (int64_t)(g.ow - 1) * g.sw + 2LL * g.dw + 1;
    if (total + 128 > (1LL << 30) || img_rows * g.n + 1024 > (1LL << 30) || (int64_t)g.h * g.w > (1LL << 28)) return false;
    if (ohw + 128 > (1LL << 22) || img_rows + 1024 > (1LL << 22)) return false;      // fast_div's range
    if (pwid > 1024 || (int64_t)g.m * g.c * kTaps + 65536 >= (1LL << 31) || g.dh > 1024) return false;
    Dense3Args& a = pl->a;
    a.n = g.n; a.c = g.c; a.h = g.h; a.w_in = g.w; a.m = g.m; a.sh = g.sh; a.sw = g.sw; a.ph = g.ph; a.pw = g.pw;
    a.dh = g.dh; a.dw = g.dw; a.oh = g.oh; a.ow = g.ow; a.act = g.act;
    pl->xvec = ids_h == 1 && ids_w == 1 && aligned16(x) && g.w % 4 == 0 && g.pw <= 4 && pwid - g.pw <= g.w + 4 ? 4 : 1;
    a.pwid = pl->xvec == 4 ? g.w + 4 : (int)pwid;
    a.col0 = pl->xvec == 4 ? 4 - g.pw : 0;
    a.img_rows = (int)img_rows; a.ids_h = ids_h; a.ids_w = ids_w; a.total_px = (int)total;
    pl->vec = aligned16(w) && (flip ? g.m : g.c) % 4 == 0 ? 4 : 1;
    double best = 0;
    int64_t best_per_cu = 0;
    bool widest = false;          // the tile of 128 pixels fits
    pl->tile = -1;
    for (int t = 0; t < kTiles; ++t) {
        if (g_force_tile >= 0 && t != g_force_tile) continue;
        const int px = 128 >> t, ch = 2 * kHalf << t;
        // rows of the stacked images that PX consecutive pixels reach; every image boundary among them adds the rows between
        const int64_t spans = (px - 1 + g.ow - 1) / g.ow + 1;
        const int64_t crossings = ohw % px == 0 ? 0 : (px - 1 + ohw - 1) / ohw;
        const int64_t rows = (spans - 1) * g.sh + 2LL * g.dh + 1 + crossings * (img_rows > (int64_t)g.oh * g.sh ? img_rows - (int64_t)g.oh * g.sh : 0);
        const int64_t rect = rows * a.pwid + (pl->xvec == 4 ? 4 : 0);     // 16-byte pieces: four zeros before the first row
        if (rect > 8192) continue;
        // the lane halves read two planes apart: half the banks. Transfers of 4 bytes fill whole wavefronts per channel
        const int64_t used = pl->xvec == 4 ? rect : ceil_div(rect, (int64_t)64) * 64;
        const int plane = (int)(ceil_div(used + 16, (int64_t)32) * 32 - 16);
        if (pl->xvec == 1 ? rect > 256 * kMaxPieces : ch * plane > 1024 * kMaxPieces * (t == 2 ? 2 : 1)) continue;
        const int x_bytes = pl->xvec == 4 ? (int)ceil_div(ch * plane, 256) * 1024 : ch * plane * 4;
        const size_t lds = 2 * ((size_t)x_bytes + weight_bytes(t, flip, pl->vec));
        if (lds > 160 * 1024) continue;
        const int64_t tiles_m = ceil_div(g.m, 32), blocks = tiles_m * ceil_div(total, (int64_t)px);
        if (blocks > kMaxBlocks) continue;
        if (t == 0) widest = true;
        const double steps = (double)ceil_div(g.c, ch);
        const int64_t per_cu = ceil_div(blocks, (int64_t)kCus);
        const double narrow = pl->xvec == 1 ? kNarrowTransfer[t] * ch * (double)ceil_div(rect, (int64_t)64) : 0.0;
        const double us = steps * fmax(kStepAlone[t] + narrow, (kStepShared[t] + narrow) * (double)per_cu) + 3.0 * ceil((double)per_cu / 3);
        if (pl->tile >= 0 && us >= best) continue;
        best = us;
        best_per_cu = per_cu;
        pl->us = us;
        pl->tile = t;
        pl->lds = lds;
        pl->blocks = (unsigned)blocks;
        a.rect = (int)rect;
        a.plane = plane;
        a.x_bytes = x_bytes;
        a.tiles_m = (int)tiles_m;
    }
    if (pl->tile < 0) return false;
    // With more than two workgroups per compute unit the general kernel is the faster one in two cases.
    // X in 4-byte pieces whose rectangles under 128 pixels do not fit, stride 2 over wide rows (32x32x113->64 74 us against 155;
    // up to two per unit 19 - 20 against 9 - 19). And one or two steps: 5 to 15 channels, unless X moves 16 bytes at a time for a
    // single tile of output channels (32x8x129->64 92 against 104, 32x8x128->64 74 against 76; 32x8x128->8 38 against 36).
    if (general && g_force_tile < 0 && best_per_cu > 2 &&
        ((pl->xvec == 1 && !widest) || (g.c > 4 && g.c < 16 && (pl->xvec == 1 || g.m > 32))))
        return false;
    return true;
}

static int launch_planned(const ConvGeom& g, int ids_h, int ids_w, bool flip, bool general, const float* x, const float* w,
                          const float* bias, float* y, hipStream_t st, const char* what, bool* applies) {
    Dense3Plan pl;
    *applies = plan_conv_dense3(g, ids_h, ids_w, flip, general, x, w, &pl);
    if (!*applies) return 0;
    note_conv_form(pl.tile);
    pl.a.x = x; pl.a.w = w; pl.a.bias = bias; pl.a.y = y;
#define DML_D3(F, V, XV) \
    if (flip == F && pl.vec == V && pl.xvec == XV) return launch_form<F, V, XV>(pl, st, what);
    DML_D3(false, 4, 4) DML_D3(false, 4, 1) DML_D3(false, 1, 4) DML_D3(false, 1, 1)
    DML_D3(true, 4, 4) DML_D3(true, 4, 1) DML_D3(true, 1, 4) DML_D3(true, 1, 1)
#undef DML_D3
    return DMLHIP_ERR_UNSUPPORTED;
}

double conv_dense3_us(const ConvGeom& g, int ids_h, int ids_w, bool flip, const void* x, const void* w, int* chains) {
    Dense3Plan pl;
    if (!plan_conv_dense3(g, ids_h, ids_w, flip, false, x, w, &pl)) return -1.0;
    *chains = 1 << pl.tile;
    return pl.us;
}

int launch_conv_dense3_f32(const ConvGeom& g, const float* x, const float* w, const float* bias, float* y, hipStream_t st,
                           bool* applies) {
    return launch_planned(g, 1, 1, false, conv_implicit_applicable(g), x, w, bias, y, st, "conv2d(dense 3x3)", applies);
}

int launch_conv_dense3_bwd_data_f32(const ConvGeom& g, const float* dy, const float* w, float* dx, hipStream_t st, bool* applies) {
    ConvGeom b;
    *applies = false;
    if (!data_gradient_problem(g, &b)) return 0;
    return launch_planned(b, g.sh, g.sw, true, conv_implicit_bwd_data_applicable(g), dy, w, nullptr, dx, st, "conv2d_backward_data(dense 3x3)", applies);
}

void conv_dense3_force_tile(int tile) { g_force_tile = tile; }

}  // namespace dml
