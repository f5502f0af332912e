// Weight gradient of a dense (group 1) 3 x 3 convolution, fp32, on v_mfma_f32_32x32x2_f32 (strides and dilations; the others on
// the bf16 matrix instructions, conv_dense3_weight_split.hip, which includes this file for the frame that both share):
//   dW[m, c, hy, hx] = sum_{n, p} dY[n, m, p] * X[n, c, oy(p) s - pad + hy d, ox(p) s - pad + hx d]
//
// What bounds it: the matrix rate, once the nine taps share what is read. A wavefront keeps the nine 32 x 32 blocks
// (channels of dY x channels of X, one per tap) in registers; a pair of pixels (split: sixteen) is one dY fragment and the shifted
// reads of the same rectangle of X for nine MFMAs (54). One workgroup of eight wavefronts per compute unit: 64 (32) channels of dY
// x 32 channels of X over a range of output rows, the wavefronts of the same channels taking every fourth (eighth) set of
// pixels. Rows of dY and the rows of X under them go global -> LDS without staging registers, a chunk of output rows of one
// image at a time, one chunk ahead, issued between the MFMAs of the chunk before. The wavefronts' sums are added through LDS
// and the ranges' results by the reduction kernel, all in a fixed order. All sums are fp32.
#include "common.h"
#include "conv_geom.h"
#include "lds_ops.h"

#include <type_traits>

namespace dml {
namespace {

constexpr int kTaps = 9, kWaves = 8, kThreads = kWaves * kWave;
constexpr int kCTile = 32;                  // channels of X per workgroup
constexpr int kMaxPixels = 512;             // of a chunk
constexpr int kCus = 256;

__device__ const floatx4 g_zeros = {0.f, 0.f, 0.f, 0.f};   // what lanes outside an operand read

struct WeightArgs {
    const float* x;
    const float* dy;
    float* part;             // [range][m][c][9]
    int n, c, h, w, m, sh, sw, ph, pw, dh, dw, oh, ow;
    int tiles_m, tiles_c, ranges;
    int rows;                // output rows of a chunk
    int pitch, plane, pwid, col0;     // LDS: floats per channel of dY and of X, per row of X, column of the padded image's column 0
    int a_bytes, x_bytes;    // LDS of a chunk's dY and X
    int a_instr, x_instr;    // transfers that fill them
};

template <int BYTES>
__device__ __forceinline__ void lds_dma(const float* gptr, char* lds_dst) {
    const auto g = (const __attribute__((address_space(1))) void*)gptr;
    const auto l = (__attribute__((address_space(3))) void*)lds_dst;
    if constexpr (BYTES == 16) __builtin_amdgcn_global_load_lds(g, l, 16, 0, 0);
    else __builtin_amdgcn_global_load_lds(g, l, 4, 0, 0);
}

struct NoSplit {
    static constexpr bool on = false;
};

struct Chunk {
    int img, oy, px;         // image, first output row, pixels
};

// WM: blocks of 32 channels of dY (1 or 2). AVEC, XVEC: floats per lane and transfer of dY and of X. SPLIT: the products on the
// bf16 matrix instructions (conv_dense3_weight_split.hip), NoSplit for the fp32 one.
template <int WM, int AVEC, int XVEC, typename SPLIT>
__device__ __forceinline__ void weight_gradient(const WeightArgs& g) {
    constexpr int MB = 32 * WM, KG = kWaves / WM;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    char* const stages = lds + kMaxPixels * 4;        // behind the pixels' offsets
    const int stage_bytes = g.a_bytes + g.x_bytes;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int l32 = lane & 31, half = lane >> 5;
    const int wm = wave % WM, kg = wave / WM;
    const int tiles = g.tiles_m * g.tiles_c;
    const int tile = blockIdx.x % (unsigned)tiles, range = blockIdx.x / (unsigned)tiles;
    const int m0 = tile % g.tiles_m * MB, c0 = tile / g.tiles_m * kCTile;
    const int total_rows = g.n * g.oh;
    int row = (int)((int64_t)total_rows * range / g.ranges);
    const int first_row = row, row_end = (int)((int64_t)total_rows * (range + 1) / g.ranges);
    const int ohw = g.oh * g.ow, in_plane = g.h * g.w;
    const float inv_pitch = 1.0f / (float)g.pitch, inv_plane = 1.0f / (float)g.plane, inv_pwid = 1.0f / (float)g.pwid;
    const uint32_t lds0 = lds_addr(lds), stages0 = lds_addr(stages);

    // byte offset of every pixel of a chunk inside a channel's rectangle of X
    for (int p = threadIdx.x; p < kMaxPixels; p += kThreads) {
        const int q = min(p, g.rows * g.ow - 1), oy = q / g.ow, ox = q - oy * g.ow;
        reinterpret_cast<int*>(lds)[p] = (oy * g.sh * g.pwid + ox * g.sw + g.col0) * 4;
    }

    auto chunk_at = [&](int r) {
        Chunk ch;
        ch.img = r / g.oh;
        ch.oy = r - ch.img * g.oh;
        ch.px = min(min(g.rows, g.oh - ch.oy), row_end - r) * g.ow;
        return ch;
    };
    // transfer i of this wavefront (the workgroup's i * 8 + wave): first those of dY, then those of X
    const int mine = (g.a_instr + g.x_instr + kWaves - 1 - wave) / kWaves;
    auto issue = [&](int i, const Chunk& ch, char* stage) {
        const int k = i * kWaves + wave;
        const float* src = reinterpret_cast<const float*>(&g_zeros);
        if (k < g.a_instr) {
            const int f = (k * kWave + lane) * AVEC;
            const int r = fast_div(f, g.pitch, inv_pitch), p = f - r * g.pitch;
            if (r < MB && m0 + r < g.m && p < ch.px)
                src = g.dy + ((int64_t)ch.img * g.m + m0 + r) * ohw + (ch.oy * g.ow + p);
            lds_dma<AVEC * 4>(src, stage + k * kWave * AVEC * 4);
        } else {
            const int f = ((k - g.a_instr) * kWave + lane) * XVEC;
            const int c = fast_div(f, g.plane, inv_plane), pos = f - c * g.plane - (XVEC == 4 ? 4 : 0);
            const int r = fast_div(max(pos, 0), g.pwid, inv_pwid);
            const int iy = ch.oy * g.sh - g.ph + r, ix = pos - r * g.pwid - (XVEC == 4 ? 0 : g.pw);
            if (c < kCTile && c0 + c < g.c && pos >= 0 && iy >= 0 && iy < g.h && ix >= 0 && ix < g.w)
                src = g.x + ((int64_t)ch.img * g.c + c0 + c) * in_plane + (iy * g.w + ix);
            lds_dma<XVEC * 4>(src, stage + g.a_bytes + (k - g.a_instr) * kWave * XVEC * 4);
        }
    };

    floatx16 acc[kTaps];
#pragma unroll
    for (int t = 0; t < kTaps; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;
    uint32_t toff[kTaps];
#pragma unroll
    for (int t = 0; t < kTaps; ++t) toff[t] = (uint32_t)((t / 3 * g.dh * g.pwid + t % 3 * g.dw) * 4);

    // the bf16 instruction loses low bits in one direction: with every other wavefront adding -dY X what is lost cancels
    const float sign = SPLIT::on && (kg & 1) ? -1.f : 1.f;

    Chunk cur = chunk_at(row);
    if (row < row_end)
        for (int i = 0; i < mine; ++i) issue(i, cur, stages);
    int stage = 0;
    while (row < row_end) {
        wait_vm_lgkm0<0>();
        __syncthreads();                 // this chunk has landed, the other stage is free
        const int next_row = row + cur.px / g.ow;
        const bool more = next_row < row_end;
        Chunk nxt = cur;
        if (more) nxt = chunk_at(next_row);
        char* const other = stages + (stage ^ 1) * stage_bytes;
        const uint32_t so = stages0 + (uint32_t)(stage * stage_bytes);
        const uint32_t a_row = so + (uint32_t)((wm * 32 + l32) * g.pitch * 4);
        const uint32_t x_row = so + (uint32_t)(g.a_bytes + l32 * g.plane * 4);
        int sent = more ? 0 : mine;
        if constexpr (SPLIT::on) {
            SPLIT::template chunk<KG>(g, acc, a_row, x_row, cur.px, kg, half, sign, [&] {
                if (sent < mine) issue(sent++, nxt, other);
            });
        } else {
            const int pairs = (cur.px + 1) / 2;
            // Pair i of pixels: 2 i in the lower lane half, 2 i + 1 in the upper. Reads run one pair ahead, the offsets two. Every
            // pair waits for what it issued and keeps it up to there: behind the last pairs of a chunk nothing multiplies what
            // was read ahead, and registers without a use would go to the transfers' addresses while the data is on its way.
            float a[2], b[2][kTaps];
            int off;
            auto read_b = [&](float (&v)[kTaps], int o) {
#pragma unroll
                for (int t = 0; t < kTaps; ++t) v[t] = lds_read_b32<0>(x_row + (uint32_t)o + toff[t]);
            };
            auto pixel = [&](int i) { return (uint32_t)(min(2 * i + half, cur.px - 1) * 4); };
            const int own = (pairs - kg + KG - 1) / KG;      // kg, kg + KG, ...
            auto pair = [&](int i, float& a_cur, float (&b_cur)[kTaps], float& a_next, float (&b_next)[kTaps]) {
                if (2 * i + 1 >= cur.px) {          // the upper half is one pixel past the chunk
                    a_cur = half ? 0.f : a_cur;
#pragma unroll
                    for (int t = 0; t < kTaps; ++t) b_cur[t] = half ? 0.f : b_cur[t];
                }
                __builtin_amdgcn_sched_barrier(0);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a_cur, b_cur[0], acc[0], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                a_next = lds_read_b32<0>(a_row + pixel(i + KG));
                read_b(b_next, off);
                off = __builtin_bit_cast(int, lds_read_b32<0>(lds0 + pixel(i + 2 * KG)));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 1; t < kTaps; ++t) {
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a_cur, b_cur[t], acc[t], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if ((t == 2 || t == 5) && sent < mine) issue(sent++, nxt, other);
                    __builtin_amdgcn_sched_barrier(0);
                }
                wait_lgkm<0>();
                __builtin_amdgcn_sched_barrier(0);
                lds_keep(a_next);
#pragma unroll
                for (int t = 0; t < kTaps; ++t) lds_keep(b_next[t]);
                lds_keep(off);
            };
            if (own > 0) {
                off = __builtin_bit_cast(int, lds_read_b32<0>(lds0 + pixel(kg)));
                const int off1 = __builtin_bit_cast(int, lds_read_b32<0>(lds0 + pixel(kg + KG)));
                a[0] = lds_read_b32<0>(a_row + pixel(kg));
                wait_lgkm<0>();
                __builtin_amdgcn_sched_barrier(0);
                read_b(b[0], off);
                wait_lgkm<0>();
                __builtin_amdgcn_sched_barrier(0);
                off = off1;
                int k = 0, i = kg;
                for (; k + 1 < own; k += 2, i += 2 * KG) {
                    pair(i, a[0], b[0], a[1], b[1]);
                    pair(i + KG, a[1], b[1], a[0], b[0]);
                }
                if (k < own) pair(i, a[0], b[0], a[1], b[1]);
            }
        }
        for (; sent < mine; ++sent) issue(sent, nxt, other);
        row = next_row;
        cur = nxt;
        stage ^= 1;
    }
    wait_vm_lgkm0<0>();

    float back = 1.f;
    if constexpr (SPLIT::on)
        back = SPLIT::template repair<KG>(g, acc, chunk_at, first_row, row_end, m0 + wm * 32 + l32, c0 + l32, kg, half, sign);

    // Eight rows of every block at a time: element e of a block is row (e / 4) * 8 + (lane / 32) * 4 + e % 4, column
    // lane % 32. The wavefronts' sums of a row are added and its 288 values written next to each other, as dW has them.
    constexpr int ROW = kCTile * kTaps + 4;
    float* const sums = reinterpret_cast<float*>(lds);
    float* const out = g.part + (int64_t)range * g.m * g.c * kTaps;
    const int cols = min(kCTile, g.c - c0) * kTaps;
#pragma unroll
    for (int eg = 0; eg < 4; ++eg) {
        __syncthreads();
#pragma unroll
        for (int t = 0; t < kTaps; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                sums[(wave * 8 + half * 4 + e) * ROW + l32 * kTaps + t] = SPLIT::on ? acc[t][eg * 4 + e] * back : acc[t][eg * 4 + e];
        __syncthreads();
        // wavefront `wave` adds row `wave` of every block
        const int m = m0 + eg * 8 + wave;
#pragma unroll
        for (int w = 0; w < WM; ++w) {
            if (m + w * 32 >= g.m) continue;
            float* const o = out + ((int64_t)(m + w * 32) * g.c + c0) * kTaps;
            const float* const s = sums + (w * 8 + wave) * ROW;
#pragma unroll
            for (int j0 = 0; j0 < kCTile * kTaps; j0 += kWave) {
                const int j = j0 + lane;
                if (j >= cols) continue;
                float v[KG / 2];
#pragma unroll
                for (int k = 0; k < KG; k += 2) v[k / 2] = s[k * WM * 8 * ROW + j] + s[(k + 1) * WM * 8 * ROW + j];
                o[j] = KG == 4 ? v[0] + v[1] : (v[0] + v[1]) + (v[KG / 2 - 2] + v[KG / 2 - 1]);
            }
        }
    }
}

template <int WM, int AVEC, int XVEC>
__global__ __launch_bounds__(kThreads) void conv_dense3_weight_kernel(const WeightArgs g) {
    weight_gradient<WM, AVEC, XVEC, NoSplit>(g);
}

struct WeightPlan {
    WeightArgs a;
    size_t lds;
};

constexpr int kLdsBytes = 160 * 1024, kSumBytes = kWaves * 8 * (kCTile * kTaps + 4) * 4;

// LDS layout of chunks of `rows` output rows; false if two of them do not fit
bool lay_out(const ConvGeom& g, int rows, int avec, int xvec, int mb, WeightPlan* pl) {
    WeightArgs& a = pl->a;
    const int64_t px = (int64_t)rows * g.ow, in_rows = (int64_t)(rows - 1) * g.sh + 2LL * g.dh + 1;
    const int64_t pwid = xvec == 4 ? g.w + 4 : (int64_t)(g.ow - 1) * g.sw + 2LL * g.dw + 1;
    const int64_t rect = in_rows * pwid + (xvec == 4 ? 4 : 0);
    if (px > kMaxPixels || rect > 16384) return false;
    // rows of 4-byte transfers an odd number of banks apart, of 16-byte transfers an odd multiple of four
    a.pitch = avec == 4 ? (int)(px / 4 | 1) * 4 : (int)px | 1;
    a.plane = xvec == 4 ? (int)(ceil_div(rect, (int64_t)4) | 1) * 4 : (int)rect | 1;
    a.pwid = (int)pwid;
    a.col0 = xvec == 4 ? 4 - g.pw : 0;
    a.rows = rows;
    a.a_instr = (int)ceil_div((int64_t)mb * a.pitch, (int64_t)kWave * avec);
    a.x_instr = (int)ceil_div((int64_t)kCTile * a.plane, (int64_t)kWave * xvec);
    a.a_bytes = a.a_instr * kWave * avec * 4;
    a.x_bytes = a.x_instr * kWave * xvec * 4;
    pl->lds = (size_t)kMaxPixels * 4 + 2 * ((size_t)a.a_bytes + a.x_bytes);
    return pl->lds <= kLdsBytes;
}

// What does not depend on the operands' addresses: whether the kernel runs and into how many ranges of output rows the
// work is cut (one workgroup per compute unit; at most 256 MiB of their results). general: another kernel takes the problem too.
int64_t plan_ranges(const ConvGeom& g, bool general) {
    if (g.kh != 3 || g.kw != 3 || g.group != 1 || g.n < 1 || g.c < 1 || g.m < 1 || g.oh < 1 || g.ow < 1) return 0;
    const int64_t per = (int64_t)g.m * g.c * kTaps, rows = (int64_t)g.n * g.oh;
    const double macs = (double)rows * g.ow * per;
    // Where the general kernel does not apply (fewer than 64 output pixels: 5x256x14x14 -> 512, stride 2, 1200 us against 35)
    // this one runs from 2^24 multiply-adds on. Where it does, the rules below hold what was measured against it, us there and
    // here: first loads, the sums through LDS and the reduction take 18 us whatever the size (1x64x56x56 -> 64 14 and 20;
    // 8x64x55x55 -> 64, 2^30, 44 and 44); channels are padded to 32, which the general kernel does
    // over all c * 9 columns (16 of 112 x 112, 64 images -> 64 1.0 - 1.16 times its time); rows of X that are no multiple of four
    // floats cost a gather per float, too much with stride 2 (64x64x113x113 -> 64 301 and 355), with
    // few multiply-adds (90 problems of 2^29 - 2^29.3: 14x64x35x35 -> 64 36 and 43, 3x64x57x57 -> 96 31 and 41, 7x32x33x33 -> 256 50 and 42; rows
    // of whole vectors 0.64 - 0.95 of its time, 1.08 at worst), with long
    // rows for a single tile of output channels (32x32x113x113 -> 32 155 and 185, -> 64 247 and 259, -> 128 525 and 492), for such a tile
    // over padded channels (times its time at 2^29.1 / 2^30.2 / 2^31 / 2^31.8: 44 of 41 x 41 -> 64 1.29 / 1.20 / 1.16 / 1.00, 24 of 33 x 33 -> 64
    // 1.17 / 1.10 / 1.07 / 1.03, 80 of 41 x 41 -> 32 1.10 / 1.11 / 1.05 / 0.88, 26 of 27 x 27 -> 32 1.06 / 0.90 / 0.83 / 0.81) or for a
    // last one that is half empty (32x96x57x57 -> 96 285 and 342).
    if (macs < (double)(1 << (general ? 29 : 24))) return 0;
    if (general) {
        const bool narrow = g.w % 4 != 0;
        const int64_t padded = ceil_div(g.c, kCTile) * kCTile;
        if (2 * padded > 3 * g.c) return 0;
        const int64_t mb = g.m > 32 ? 64 : 32;
        if (narrow && (g.sw > 1 || (g.ow > 64 && g.m <= 64) || 4 * ceil_div(g.m, mb) * mb > 5 * g.m)) return 0;
        if (narrow && g.m < 128 && macs < 7.0e8) return 0;
        // columns here for one there
        const double columns = (double)(padded * kTaps) / (double)(ceil_div((int64_t)g.c * kTaps, (int64_t)32) * 32);
        const double least = columns > 1.35 ? 1e18 : columns > 1.2 ? (g.ow < 50 ? 3.0e9 : 1e18) : columns > 1.15 ? 2.2e9 : 1.1e9;
        if (narrow && g.m <= 64 && columns > 1.0 && macs < least) return 0;
    }
    if (rows > (1LL << 30) || per > (1LL << 30) || (int64_t)g.oh * g.ow > (1LL << 28) || (int64_t)g.h * g.w > (1LL << 28)) return 0;
    WeightPlan pl;
    if (!lay_out(g, 1, 1, 1, g.m > 32 ? 64 : 32, &pl)) return 0;
    const int64_t tiles = ceil_div(g.m, g.m > 32 ? 64 : 32) * ceil_div(g.c, kCTile);
    int64_t ranges = kCus / tiles;
    const int64_t cap = (64LL << 20) / per;
    if (ranges > cap) ranges = cap;
    if (ranges > rows) ranges = rows;
    if (ranges < 1) ranges = 1;
    return ranges * tiles <= 2147483647LL ? ranges : 0;
}

int launch_weight(void (*kern)(const WeightArgs), const WeightPlan& pl, unsigned blocks, hipStream_t st) {
    const size_t lds = pl.lds > (size_t)kSumBytes ? pl.lds : (size_t)kSumBytes;
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
        set_error("conv2d_backward_weight: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        return (int)e;
    }
    hipLaunchKernelGGL(kern, blocks, kThreads, lds, st, pl.a);
    return launch_status("conv2d_backward_weight(dense 3x3)");
}

bool plan_weight(const ConvGeom& g, const void* x, const void* dy, WeightPlan* pl, unsigned* blocks, int* avec, int* xvec) {
    const int64_t ranges = plan_ranges(g, false);
    if (ranges < 1) return false;
    const int mb = g.m > 32 ? 64 : 32;
    *avec = g.ow % 4 == 0 && aligned16(dy) ? 4 : 1;
    *xvec = g.w % 4 == 0 && aligned16(x) && g.pw <= 4 && (int64_t)(g.ow - 1) * g.sw + 2LL * g.dw - g.pw < g.w + 4 ? 4 : 1;
    if (!lay_out(g, 1, *avec, *xvec, mb, pl)) *avec = *xvec = 1;
    WeightArgs& a = pl->a;
    a.n = g.n; a.c = g.c; a.h = g.h; a.w = g.w; a.m = g.m; a.sh = g.sh; a.sw = g.sw; a.ph = g.ph; a.pw = g.pw;
    a.dh = g.dh; a.dw = g.dw; a.oh = g.oh; a.ow = g.ow;
    a.tiles_m = (int)ceil_div(g.m, mb);
    a.tiles_c = (int)ceil_div(g.c, kCTile);
    a.ranges = (int)ranges;
    // as many rows as fit, but no more than split a range (and an image) into equal chunks
    int most = 1;
    const int64_t range_rows = ceil_div((int64_t)g.n * g.oh, ranges);
    const int limit = range_rows < g.oh ? (int)range_rows : g.oh;
    while (most < limit && lay_out(g, most + 1, *avec, *xvec, mb, pl)) ++most;
    const int rows = (int)ceil_div(limit, ceil_div(limit, most));
    if (!lay_out(g, rows, *avec, *xvec, mb, pl)) return false;
    *blocks = (unsigned)(ranges * a.tiles_m * a.tiles_c);
    return true;
}

}  // namespace

int64_t conv_dense3_bwd_weight_partials(const ConvGeom& g, bool general) { return plan_ranges(g, general); }

int launch_conv_dense3_bwd_weight(const ConvGeom& g, const float* x, const float* dy, float* part, hipStream_t st) {
    WeightPlan pl;
    unsigned blocks;
    int avec, xvec;
    DML_REQUIRE(plan_weight(g, x, dy, &pl, &blocks, &avec, &xvec), DMLHIP_ERR_UNSUPPORTED,
                "conv2d_backward_weight: the 3x3 kernel does not apply");
    pl.a.x = x; pl.a.dy = dy; pl.a.part = part;
    const int wm = g.m > 32 ? 2 : 1;
#define DML_D3W(WM, AV, XV) \
    if (wm == WM && avec == AV && xvec == XV) return launch_weight(conv_dense3_weight_kernel<WM, AV, XV>, pl, blocks, st);
    DML_D3W(1, 1, 1) DML_D3W(1, 1, 4) DML_D3W(1, 4, 1) DML_D3W(1, 4, 4)
    DML_D3W(2, 1, 1) DML_D3W(2, 1, 4) DML_D3W(2, 4, 1) DML_D3W(2, 4, 4)
#undef DML_D3W
    return DMLHIP_ERR_UNSUPPORTED;
}

}  // namespace dml
