// Dense (group 1) 3 x 3 convolution, fp32, on the bf16 matrix instructions: the forward pass and, with the weights read
// transposed and reversed, the data gradient. Operands are split into three bf16 values each (bf16_split.h).
//   Y[n, m, p] = act(b[m] + sum_{c, hy, hx} W[m, c, hy, hx] * X[n, c, oy(p) s - pad + hy d, ox(p) s - pad + hx d])
//
// A workgroup of eight wavefronts computes 64 output channels x 128 P pixels, counted through the batch; a wavefront 32 channels
// x 32 P pixels. A step is 16 input channels: the weights of the step and the rectangle of X under the tile's pixels go from
// global memory into registers, are split once, and lie in LDS as chunks of eight channels of one bf16 value, so that a fragment
// of an MFMA is one 16-byte read and every tap a shifted read of the same rectangle. The next step's values are loaded and
// split while this step's products run.
//
// What bounds it: the matrix pipe in the products (P = 4: 7.1 us per step, 6.5 at its rate; LDS is read at 0.6 - 1.0 of its rate),
// the loads of the chunks beside them (1 us per step: 8 loads of 4 bytes per lane for a chunk; with the loads left out P = 4 takes
// 7.3 us, P = 1 2.5 of 3.2), 0.5 us for the stores to LDS and the barriers, and per tile 5 us of first loads and 3 - 9 us of
// results, which one workgroup per compute unit does not hide. Measured, us forward / data gradient, the kernel of
// conv_dense3.hip and here: 32x64x56x56 -> 64 82 / 80 and 54 / 54, 32x64x56x56 -> 128 144 / 150 and 104 / 90, 32x128x28x28 -> 128
// 84 / 83 and 65 / 63, 32x256x14x14 -> 256 107 / 105 and 58 / 56. What the products waited for until it was changed: 64 copies of the
// activation in the epilogue (12 us per tile), loads behind branches (their addresses in 64 registers, 2 us per step).
//
// The large product h h has a sum of its own (P = 1: two), so that the roundings of the five small ones are not roundings of the
// result: 2 of these for sixteen products instead of 12. Error against fp64 as a share of that of the fp32 instruction (one sum for P = 2 and
// 4, two for P = 1; 16 - 2048 channels; with all six products in one sum in brackets): normal operands 0.31 - 0.41 (0.83 - 0.87), X
// behind a ReLU 0.34 - 0.52 (1.08 - 1.20), nothing negative 0.27 - 0.62 (0.9 - 1.7). None takes more than 1 - 2 % longer for it. (P = 4
// has registers for two such sums. Added after every tap, and not once per step and pair of blocks, they took 5 us of 32x64x56x56 -> 64.)
#include "bf16_split.h"
#include "conv_geom.h"

#include <type_traits>

namespace dml {
namespace {

constexpr int kTaps = 9;
constexpr int kThreads = 512;
constexpr int kRows = 64;                    // output channels of a tile
constexpr int kCh = 16;                      // input channels of a step
constexpr int kCus = 256, kXcds = 8;
constexpr int kWChunks = 2 * kTaps + 1;      // 16-byte chunks per output channel: an odd number, so that fragments of 32 channels do not conflict
constexpr int kWPlane = kRows * kWChunks * 16, kWBytes = 3 * kWPlane;
constexpr int kWTasks = kRows * 2 * kTaps;    // chunks of a step's weights: whole wavefronts
constexpr int kMaxLds = 160 * 1024;
constexpr uint32_t kZeros = 0x80000000u;     // buffer offset past the end of every buffer: loads return zero
constexpr int kBufferFlags = 0x00020000;     // raw buffer of 32-bit data

struct SplitArgs3 {
    const float* x;
    const float* w;
    const float* bias;
    float* y;
    int n, c, h, w_in, m, sh, sw, ph, pw, dh, dw, oh, ow, act;
    int img_rows;             // rows of a padded image: rectangles are cut from the images stacked on each other
    int pwid, rect;           // rectangle columns and positions
    int ids_h, ids_w;         // data gradient: dY is read as if ids - 1 zeros stood between its rows / columns
    int total_px, tiles_m;
    unsigned blocks;
};

template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

template <bool FLIP>
__device__ __forceinline__ int64_t weight_at(const SplitArgs3& g, int m, int c, int tap) {
    return FLIP ? ((int64_t)c * g.m + m) * kTaps + (kTaps - 1 - tap) : ((int64_t)m * g.c + c) * kTaps + tap;
}

// P: blocks of 32 pixels per wavefront. TASKS: chunks per thread and step.
template <int P, int TASKS, bool FLIP>
__global__ __launch_bounds__(kThreads, 2) void conv_dense3_split_kernel(const SplitArgs3 g) {
    constexpr int PX = 128 * P;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    char* const xs = lds + kWBytes;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int l32 = lane & 31, half = lane >> 5;
    const int wm = wave >> 2, wp = wave & 3;
    unsigned bid = blockIdx.x;
    {
        const unsigned xcd = bid % kXcds, idx = bid / kXcds, base = g.blocks / kXcds, rem = g.blocks % kXcds;
        bid = xcd * base + (xcd < rem ? xcd : rem) + idx;
    }
    const int m0 = (int)(bid % (unsigned)g.tiles_m) * kRows;
    const int p0 = (int)(bid / (unsigned)g.tiles_m) * PX;
    const int ohw = g.oh * g.ow;
    const float inv_ohw = 1.0f / (float)ohw, inv_ow = 1.0f / (float)g.ow, inv_rows = 1.0f / (float)g.img_rows;
    const float inv_pwid = 1.0f / (float)g.pwid, inv_rect = 1.0f / (float)g.rect;

    // pixel p of the batch reads row n img_rows + oy sh + hy dh of the stacked images, column ox sw + hx dw
    const int n_first = p0 / ohw, q_first = p0 - n_first * ohw;
    const int r_first = q_first / g.ow * g.sh;        // in its image
    const int xplane = 2 * g.rect * 16;               // bytes of one bf16 value of the rectangle
    int xaddr[P];                                     // this lane's pixel of block j at tap 0
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int p = p0 + (wp * P + j) * 32 + l32;
        const int q0 = min(p, g.total_px - 1) - p0 + q_first;
        const int n = fast_div(q0, ohw, inv_ohw), q = q0 - n * ohw;
        const int oy = fast_div(q, g.ow, inv_ow), ox = q - oy * g.ow;
        xaddr[j] = (half * g.rect + (n * g.img_rows + oy * g.sh - r_first) * g.pwid + ox * g.sw) * 16;
    }
    const int waddr = ((wm * 32 + l32) * kWChunks + half * kTaps) * 16;

    // What this thread brings in: chunks of eight channels, of a tap of an output channel (the first kWTasks) or at a position of
    // the rectangle. Buffer loads: byte offset of the chunk from channel 0 of the weights or of image n_first, kZeros (past the
    // end of either) where there is nothing to read. `late`: chunks of the upper eight channels of a step.
    const int in_plane = g.h * g.w_in;
    // row and column of the padded image n_first + n, channel c
    auto x_offset = [&](int n, int row, int col, int c) -> uint32_t {
        int iy = row - g.ph, ix = col - g.pw;
        bool ok = iy >= 0 && ix >= 0;
        if (g.ids_h > 1 || g.ids_w > 1) {
            const int qy = max(iy, 0) / g.ids_h, qx = max(ix, 0) / g.ids_w;
            ok = ok && qy * g.ids_h == iy && qx * g.ids_w == ix;
            iy = qy;
            ix = qx;
        }
        ok = ok && iy < g.h && ix < g.w_in;
        return ok ? (uint32_t)((n * g.c + c) * in_plane + iy * g.w_in + ix) * 4 : kZeros;
    };
    const int wstep = (FLIP ? g.m : 1) * kTaps;        // elements from one channel to the next
    uint32_t off[TASKS], late = 0;
#pragma unroll
    for (int u = 0; u < TASKS; ++u) {
        const int first = u * kThreads + wave * kWave;
        int kh;
        if (first < kWTasks) {
            const int task = first + lane, m = task / (2 * kTaps), k = task - m * 2 * kTaps;
            kh = k / kTaps;
            off[u] = m0 + m < g.m ? (uint32_t)(weight_at<FLIP>(g, m0 + m, 8 * kh, k - kh * kTaps) * 4) : kZeros;
        } else {
            const int task = first + lane - kWTasks;
            kh = fast_div(task, g.rect, inv_rect);
            const int pos = task - kh * g.rect, row = fast_div(pos, g.pwid, inv_pwid);
            const int n = fast_div(r_first + row, g.img_rows, inv_rows);
            off[u] = kh < 2 && n_first + n < g.n ? x_offset(n, r_first + row - n * g.img_rows, pos - row * g.pwid, 8 * kh) : kZeros;
        }
        late |= kh == 1 ? 1u << u : 0u;
    }
    const int64_t x_left = (int64_t)(g.n - n_first) * g.c * in_plane * 4;
    const auto xbuf = __builtin_amdgcn_make_buffer_rsrc((void*)(g.x + (int64_t)n_first * g.c * in_plane), 0,
                                                        (int)min(x_left, (int64_t)0x7fffffff), kBufferFlags);
    const auto wbuf = __builtin_amdgcn_make_buffer_rsrc((void*)g.w, 0, g.m * g.c * kTaps * 4, kBufferFlags);
    float raw[TASKS][8];
    auto load = [&](int u, int c0) {
        const bool weights = u * kThreads + wave * kWave < kWTasks;
        const int step = weights ? wstep : in_plane;
        const auto buf = weights ? wbuf : xbuf;
        // channels come in eights: the last step may have the lower ones only
        const uint32_t o = c0 + 8 >= g.c && (late >> u & 1) ? kZeros : off[u];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            raw[u][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buf, o, (c0 + e) * step * 4, 0));
    };
    Pieces pieces[TASKS];
    auto store = [&] {
#pragma unroll
        for (int u = 0; u < TASKS; ++u) {
            const int task = u * kThreads + (int)threadIdx.x;
            const bool weights = u * kThreads + wave * kWave < kWTasks;
            if (!weights && task - kWTasks >= 2 * g.rect) continue;
            const int plane = weights ? kWPlane : xplane;
            char* const p = lds + (weights ? task + task / (2 * kTaps) * (kWChunks - 2 * kTaps) : kWBytes / 16 + task - kWTasks) * 16;
            *reinterpret_cast<bf16x8*>(p) = pieces[u].h;
            *reinterpret_cast<bf16x8*>(p + plane) = pieces[u].m;
            *reinterpret_cast<bf16x8*>(p + 2 * plane) = pieces[u].l;
        }
    };

    floatx16 acc[P];
#pragma unroll
    for (int j = 0; j < P; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
    floatx16 odd;                                              // P = 1: a second sum, of the odd taps
#pragma unroll
    for (int e = 0; e < 16; ++e) odd[e] = 0.f;
    // Sums of the small products. P = 1 and 2 keep them to the end; P = 4 has registers for two and takes its blocks in two passes over the
    // taps of a step, which add them to acc.
    constexpr int PASSES = P == 4 ? 2 : 1, B = P / PASSES;
    floatx16 low[B];
#pragma unroll
    for (int j = 0; j < B; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) low[j][e] = 0.f;

    auto weights_at = [&](int tap) -> Pieces {
        const char* const p = lds + waddr + tap * 16;
        return {*reinterpret_cast<const bf16x8*>(p), *reinterpret_cast<const bf16x8*>(p + kWPlane),
                *reinterpret_cast<const bf16x8*>(p + 2 * kWPlane)};
    };
    auto pixels_at = [&](int j, int tap) -> Pieces {
        const char* const p = xs + xaddr[j] + (tap / 3 * g.dh * g.pwid + tap % 3 * g.dw) * 16;
        return {*reinterpret_cast<const bf16x8*>(p), *reinterpret_cast<const bf16x8*>(p + xplane),
                *reinterpret_cast<const bf16x8*>(p + 2 * xplane)};
    };
    // The products of a step. Fragments are read one block ahead; SPLIT: the chunks of the next step are split under the
    // products. Where registers allow, their values are loaded a step ahead, as soon as the registers are free (at the start
    // of the step that splits them, 1 us of it was a wait); elsewhere when the step begins, and are split under the last taps.
    constexpr bool AHEAD = P < 4 && TASKS < 7;
    auto step = [&](int next, auto split_c) {                  // next: first channel of the chunks that are loaded
        constexpr bool SPLIT = decltype(split_c)::value;
        Pieces a[2], b[2];
        a[0] = weights_at(0);
        b[0] = pixels_at(0, 0);
        static_for<0, kTaps * PASSES>([&](auto tc) {
            constexpr int at = decltype(tc)::value, tap = at % kTaps, pass = at / kTaps, u = at - (kTaps * PASSES - TASKS);
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, B>([&](auto jc) {
                constexpr int j = decltype(jc)::value, i = at * B + j, n = i + 1;
                if constexpr (n < kTaps * P) {
                    if constexpr (j + 1 == B) a[(at + 1) & 1] = weights_at((at + 1) % kTaps);
                    b[n & 1] = pixels_at(n / B / kTaps * B + n % B, n / B % kTaps);
                }
                floatx16& large = P == 1 && tap % 2 ? odd : acc[pass * B + j];
                large = mfma_large(a[at & 1], b[i & 1], large);
                low[j] = mfma_small(a[at & 1], b[i & 1], P == 4 && tap == 0 ? floatx16{} : low[j]);
                if constexpr (P == 4 && tap + 1 == kTaps) {
                    acc[pass * B + j] += low[j];
                    asm volatile("" : "+v"(acc[pass * B + j]));
                }
            });
            if constexpr (SPLIT && u >= 0) pieces[u] = split_eight(raw[u]);
#pragma unroll
            for (int i = 0; i < 6 * B; ++i) {       // a matrix instruction, then what can issue under it
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, P == 1 ? 9 : P == 2 ? 4 : 5, 0);
            }
            if constexpr (SPLIT && u >= 0) {
                asm volatile("" : "+v"(pieces[u].h), "+v"(pieces[u].m), "+v"(pieces[u].l));   // computed here, not at the stores
                if constexpr (AHEAD) load(u, next);
            }
        });
        __builtin_amdgcn_sched_barrier(0);
    };

#pragma unroll
    for (int u = 0; u < TASKS; ++u) load(u, 0);
#pragma unroll
    for (int u = 0; u < TASKS; ++u) pieces[u] = split_eight(raw[u]);
    store();
    const int last = (g.c - 1) / kCh * kCh;
    if constexpr (AHEAD) {
#pragma unroll
        for (int u = 0; u < TASKS; ++u) load(u, min(kCh, last));
    }
    __syncthreads();
    for (int c0 = 0; c0 < last; c0 += kCh) {
        if constexpr (!AHEAD) {
#pragma unroll
            for (int u = 0; u < TASKS; ++u) load(u, c0 + kCh);
        }
        step(min(c0 + 2 * kCh, last), std::true_type{});
        __syncthreads();
        store();
        __syncthreads();
    }
    step(0, std::false_type{});
    if constexpr (P == 1) acc[0] += odd;
    if constexpr (P < 4) {
#pragma unroll
        for (int j = 0; j < P; ++j) acc[j] += low[j];
    }

    // What follows finds its pixels again: addresses kept from the start would be registers that the loop does not have.
    int tid = threadIdx.x, pixels = ohw;
    asm volatile("" : "+v"(tid), "+s"(pixels));
    const int row32 = tid & 31, upper = tid >> 5 & 1;
    const float inv_pixels = 1.0f / (float)pixels;
    const int first = p0 + wp * P * 32 + row32;         // this lane's pixel of block 0

    // A value without a split (infinite, NaN, from 2^112 on) makes a sum that is not finite: this wavefront's sums once more,
    // on the fp32 instruction (32x64x56x56 -> 64 with NaN in one pixel / everywhere: one such product 12.0 / 10.5 ms when every lane did
    // its sums one after the other).
    float bad = 0.f;
#pragma unroll
    for (int j = 0; j < P; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) bad = __builtin_fmaf(acc[j][e], 0.f, bad);
    if (__builtin_amdgcn_ballot_w64(bad != 0.f) != 0) {
#pragma unroll
        for (int j = 0; j < P; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
        const int m = m0 + wm * 32 + row32;
#pragma unroll 1
        for (int tap = 0; tap < kTaps; ++tap) {
            // of channel `upper`: the instruction takes two, one per lane half
            const uint32_t woff = m < g.m ? (uint32_t)(weight_at<FLIP>(g, m, upper, tap) * 4) : kZeros;
            uint32_t xoff[P];
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const int q0 = min(first + j * 32, g.total_px - 1) - n_first * pixels;
                const int n = fast_div(q0, pixels, inv_pixels), q = q0 - n * pixels, oy = q / g.ow;
                xoff[j] = x_offset(n, oy * g.sh + tap / 3 * g.dh, (q - oy * g.ow) * g.sw + tap % 3 * g.dw, upper);
            }
#pragma unroll 1
            for (int c = 0; c < g.c; c += 8) {      // channels come in eights
                float a[4], b[4][P];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    a[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wbuf, woff, (c + 2 * i) * wstep * 4, 0));
#pragma unroll
                    for (int j = 0; j < P; ++j)
                        b[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, xoff[j], (c + 2 * i) * in_plane * 4, 0));
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < P; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i][j], acc[j], 0, 0, 0);
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < P; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][e] *= kSplitBack;
    }

    // element e of a block: row (e / 4) * 8 + (lane / 32) * 4 + e % 4, column lane % 32
    const int mw = m0 + wm * 32 + upper * 4;
    float b[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int m = mw + (e >> 2) * 8 + (e & 3);
        b[e] = g.bias && m < g.m ? g.bias[m] : 0.f;
    }
    // The activation in the loop is none or ReLU. The others are applied behind it to what was stored, in a loop that is not
    // unrolled: 16 P copies of them do not fit the instruction cache (P = 4: 12 us per tile for the stores alone).
    const bool relu = g.act == DMLHIP_ACT_RELU;
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int p = first + j * 32;
        if (p >= g.total_px) continue;
        const int n = fast_div(p - n_first * pixels, pixels, inv_pixels), q = p - (n_first + n) * pixels;
        float* const out = g.y + ((int64_t)(n_first + n) * g.m + mw) * pixels + q;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int r = (e >> 2) * 8 + (e & 3);
            const float v = acc[j][e] + b[e];       // NaN of a bias stays NaN but under ReLU
            if (mw + r < g.m) out[(int64_t)r * pixels] = relu ? fmaxf(v, 0.f) : v;
        }
    }
    if (g.act != DMLHIP_ACT_NONE && g.act != DMLHIP_ACT_RELU) {
        for (int j = 0; j < P; ++j) {
            const int p = first + j * 32;
            if (p >= g.total_px) continue;
            const int n = p / pixels, q = p - n * pixels;
            float* const out = g.y + ((int64_t)n * g.m + mw) * pixels + q;
#pragma unroll 1
            for (int e = 0; e < 16; ++e) {
                const int r = (e >> 2) * 8 + (e & 3);
                if (mw + r < g.m) out[(int64_t)r * pixels] = apply_act(g.act, out[(int64_t)r * pixels]);
            }
        }
    }
}

struct SplitPlan3 {
    SplitArgs3 a;
    int p, tasks;
    size_t lds;
};

template <int P, int TASKS, bool FLIP>
int launch(const SplitPlan3& pl, hipStream_t st, const char* what) {
    auto kern = conv_dense3_split_kernel<P, TASKS, FLIP>;
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds);
    if (e != hipSuccess) {
        set_error("%s: cannot reserve %zu bytes of LDS: %s", what, pl.lds, hipGetErrorString(e));
        return (int)e;
    }
    note_conv_form(P == 1 ? (TASKS == 4 ? 3 : TASKS == 6 ? 11 : 19) : P == 2 ? (TASKS == 5 ? 4 : 12) : TASKS == 6 ? 5 : 13);
    hipLaunchKernelGGL(kern, pl.a.blocks, kThreads, pl.lds, st, pl.a);
    return launch_status(what);
}

template <bool FLIP>
int launch_form(const SplitPlan3& pl, hipStream_t st, const char* what) {
    if (pl.p == 1 && pl.tasks > 4) return pl.tasks <= 6 ? launch<1, 6, FLIP>(pl, st, what) : launch<1, 7, FLIP>(pl, st, what);
    if (pl.p == 1) return launch<1, 4, FLIP>(pl, st, what);
    if (pl.p == 2) return pl.tasks <= 5 ? launch<2, 5, FLIP>(pl, st, what) : launch<2, 7, FLIP>(pl, st, what);
    return pl.tasks <= 6 ? launch<4, 6, FLIP>(pl, st, what) : launch<4, 7, FLIP>(pl, st, what);
}

thread_local int g_last_form = -1;   // diagnostic
thread_local int g_force_p = 0;     // diagnostic: blocks of 32 pixels per wavefront (0 = chosen here); -1: not this kernel

}  // namespace

// The geometry is the product's own: for a data gradient the stride-1 convolution of the (zero-dilated) dY. *us: estimated time.
static bool plan_split(const ConvGeom& g, int ids_h, int ids_w, int most_p, SplitPlan3* pl, double* us) {
    if (g_force_p < 0 || g.kh != 3 || g.kw != 3 || g.group != 1 || g.n < 1 || g.c < 16 || g.c % 8 || g.m < 1 || g.oh < 1 || g.ow < 1) return false;
    const int64_t ohw = (int64_t)g.oh * g.ow, total = (int64_t)g.n * ohw;
    const int64_t img_rows = (int64_t)(g.oh - 1) * g.sh + 2LL * g.dh + 1, pwid = (int64_t)(g.ow - 1) * g.sw + 2LL * g.dw + 1;
    if (total + 1024 > (1LL << 30) || img_rows * g.n + 4096 > (1LL << 30) || ohw + 1024 > (1LL << 22) || img_rows + 4096 > (1LL << 22))
        return false;                                                                        // fast_div's range
    if (pwid > 1024 || g.dh > 1024 || (int64_t)g.m * g.c * kTaps > (1LL << 28)) return false;
    pl->p = 0;
    for (int p = 1; p <= most_p; p *= 2) {
        if (g_force_p > 0 && p != g_force_p) continue;
        const int64_t px = 128LL * p;
        // rows of the stacked images that PX consecutive pixels reach; every image boundary among them adds the rows between
        const int64_t spans = (px - 1 + g.ow - 1) / g.ow + 1;
        const int64_t crossings = ohw % px == 0 ? 0 : (px - 1 + ohw - 1) / ohw;
        const int64_t between = img_rows > (int64_t)g.oh * g.sh ? img_rows - (int64_t)g.oh * g.sh : 0;
        const int64_t rows = (spans - 1) * g.sh + 2LL * g.dh + 1 + crossings * between, rect = rows * pwid;
        if (kWBytes + rect * 96 > kMaxLds) continue;
        if ((crossings + 1) * (double)g.c * g.h * g.w > (double)(1 << 29)) continue;          // 31-bit offsets inside a tile
        const int64_t tiles_m = ceil_div(g.m, (int64_t)kRows), blocks = tiles_m * ceil_div(total, px);
        if (blocks > (1LL << 22)) continue;
        const double steps = (double)ceil_div(g.c, (int64_t)kCh), rounds = (double)ceil_div(blocks, (int64_t)kCus);
        // us of a tile: first loads and results, and per step; whole rounds of one tile per compute unit. Rounds decide: 32x64x56x56 ->
        // 64 is one round of 196 tiles of 512 pixels (54 us), two of 392 (58) or four (92), 32x256x14x14 -> 256 one of 196 tiles of 128
        // (58; of 256 81, of 512 154).
        // More chunks per thread, larger rectangles, take longer (18 shapes, strides, dilation, 28 - 112 pixels wide).
        const int tasks = (int)ceil_div(kWTasks + 2 * rect, (int64_t)kThreads);
        const double step = p == 1 ? (tasks <= 4 ? 3.4 : tasks <= 6 ? 4.1 : 4.9) : p == 2 ? (tasks <= 5 ? 4.9 : 6.0) : tasks <= 6 ? 8.9 : 10.2;
        const double t = rounds * ((p == 1 ? 7.0 : p == 2 ? 9.0 : steps > 1 ? 15.0 : 12.0) + step * steps);
        if (pl->p > 0 && t >= *us) continue;
        *us = t;
        pl->p = p;
        pl->tasks = tasks;
        pl->lds = (size_t)(kWBytes + rect * 96);
        SplitArgs3& a = pl->a;
        a.n = g.n; a.c = g.c; a.h = g.h; a.w_in = g.w; a.m = g.m; a.sh = g.sh; a.sw = g.sw; a.ph = g.ph; a.pw = g.pw;
        a.dh = g.dh; a.dw = g.dw; a.oh = g.oh; a.ow = g.ow; a.act = g.act;
        a.img_rows = (int)img_rows; a.pwid = (int)pwid; a.rect = (int)rect;
        a.ids_h = ids_h; a.ids_w = ids_w; a.total_px = (int)total; a.tiles_m = (int)tiles_m; a.blocks = (unsigned)blocks;
    }
    return pl->p > 0;
}

static int launch_split(const ConvGeom& g, int ids_h, int ids_w, bool flip, const float* x, const float* w, const float* bias, float* y,
                        hipStream_t st, const char* what, bool* applies) {
    SplitPlan3 pl;
    double us;
    // No larger errors than the kernel on the fp32 instruction would have, whatever the operands. P = 2 and 4 have 0.37 - 0.62 of those of its
    // one sum, up to 1.01 and 1.23 of those of two (nothing negative), P = 1 0.27 - 0.53 of those of two; of four none is as exact everywhere.
    int chains = 1;
    double other = 0;
    if (g_force_p == 0) {
        other = conv_dense3_us(g, ids_h, ids_w, flip, x, w, &chains);
        *applies = other > 0 && chains <= 2;
        if (!*applies) return 0;
    }
    *applies = plan_split(g, ids_h, ids_w, chains == 2 ? 1 : 4, &pl, &us);
    if (*applies && g_force_p == 0) *applies = us < other;
    if (!*applies) return 0;
    pl.a.x = x; pl.a.w = w; pl.a.bias = bias; pl.a.y = y;
    return flip ? launch_form<true>(pl, st, what) : launch_form<false>(pl, st, what);
}

int launch_conv_dense3_split_f32(const ConvGeom& g, const float* x, const float* w, const float* bias, float* y, hipStream_t st,
                                 bool* applies) {
    return launch_split(g, 1, 1, false, x, w, bias, y, st, "conv2d(dense 3x3)", applies);
}

int launch_conv_dense3_split_bwd_data_f32(const ConvGeom& g, const float* dy, const float* w, float* dx, hipStream_t st, bool* applies) {
    ConvGeom b;
    *applies = false;
    if (!data_gradient_problem(g, &b)) return 0;
    return launch_split(b, g.sh, g.sw, true, dy, w, nullptr, dx, st, "conv2d_backward_data(dense 3x3)", applies);
}

void note_conv_form(int form) { g_last_form = form; }

}  // namespace dml

extern "C" int dmlhip_debug_last_conv_form(void) {
    const int form = dml::g_last_form;
    dml::g_last_form = -1;
    return form;
}

extern "C" void dmlhip_debug_force_conv_dense3_tile(int tile) {
    dml::g_force_p = tile < 0 ? 0 : tile < 3 ? -1 : 1 << (tile - 3);
    dml::conv_dense3_force_tile(tile < 3 ? tile : -1);
}
