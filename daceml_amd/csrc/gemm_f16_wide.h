// fp16 GEMM for products of many 256 x 256 tiles: one workgroup of four wavefronts per compute unit that stays for all of
// its tiles, v_mfma_f32_16x16x32_f16, both operands straight from global memory into LDS (buffer_load ... lds). The same with
// 128 x 128 tiles and twice as many steps on their way, where products have fewer. What follows is about the large tile.
//
// What bounds it: the matrix pipe at the clock that the power limit leaves (1.4 - 1.6 GHz under this load). A 64-k step of a
// wavefront is 128 MFMAs = 2048 clocks and takes 2240 - 2290; the 256 x 256 tile of gemm_f16_pipe.h takes 2550 - 2650 with
// 32 x 32 x 16 instructions, which also draw more power for the same product (1.31 against 1.40 GHz measured side by side).
// What it does differently, each measured on its own:
//  * The transfers of a step are spread over the whole of it, one after every eighth MFMA. They move 64 bytes per clock and
//    compute unit: issued in half of the step's time they queue up, and the wavefront that waits to issue the next one
//    issues no MFMA (2550 clocks with two stages of both operands and half a step to refill one, 2330 where all of them
//    go out in the last half with every fourth MFMA). 160 KB of LDS hold two tiles of A and three of B: B's tile of step
//    t + 2 goes out in the first half of step t (its stage has been free since step t - 1), A's in the second half (its stage
//    is the one whose last fragments were just read), and every transfer has at least half a step to land.
//  * buffer_load takes a 32-bit offset per lane and a scalar one: no 64-bit address is formed per lane and transfer.
//  * A workgroup keeps the transfers running across its tiles: the first two steps of its next tile are on their way while it
//    writes a tile, so only the first tile of a launch waits for memory (2.1 - 2.8 us).
//  * The accumulators go to memory without LDS (wide_epilogue). With the operands swapped (B first) lane l holds row l % 16
//    and columns 4 (l / 16) .. + 3 of a 16 x 16 block.
// The MFMAs are inline assembly with the accumulator tied to an accumulation register: the compiler moves 2 - 9 of the 64
// accumulators between register files in every step otherwise (2400 against 2270 clocks).
//
// The 128 x 128 tile is bound by the L2s: 32 KB per 64 k and compute unit, 512 clocks of the 64 bytes that one gets at best, all
// 256 together 18 - 19 TB/s of a step's 0.44 us (0.50 in gemm_f16_pipe.h). 4096 x 1024 x 4096 with residual 39.8 -> 36.7 us, B
// row-contiguous 39.6 -> 36.3, three pairs of 4096 x 1024 x 1024 33.5 -> 30.2, 8192 x 1024 x 4096 75 -> 69.
//
// LDS tiles. KC (K contiguous): [256 rows][64 k], 128-byte rows, 16-byte chunk c of row r at slot c ^ (r & 7) ^ (r >> 3 & 1).
// RC (rows contiguous): [64 k][256 rows], chunk c (8 rows) of K row k at slot c ^ ((k & 3) << 2) ^ ((k >> 3 & 1) << 1): the
// transpose read of 16 lanes touches four K rows, 32 bytes of each, the two groups that are read together are eight K rows
// apart. LDS clocks: a KC fragment 8, four of them bank conflicts (the 32-row fragments of gemm_f16_pipe.h have none), an RC one of A
// twice 2 without conflicts, one of B, whose columns b_row moves, twice 4. All reads of a step take half as long as its MFMAs.
//  * SLICED (weight gradients: few tiles, a long K): the workgroups of a tile share its K steps and write fp32 partial results
//    that wide_sum_kernel adds up, four times over for 64 tiles: 64 MB written and read, about 30 us whatever K is. The row
//    sums of A (the bias gradient) are taken from the fragments: the workgroups of tile column c add those of every step that
//    leaves c modulo the number of columns, so that none of them falls behind the others. Any K: the step with its last k is
//    sent by a copy of the step of its own, with zeros behind them.
// Requirements (checked by the host): K % 64 == 0 (but for SLICED), more steps than are ahead (three of the large tile, five of the
// small one, those of all operand pairs together), no activation, beta == 0, n % 8 == 0, 16-byte aligned operands, column bias and
// result rows, 32-bit element offsets, rows % 8 == 0 for RC operands.
#pragma once

#include "gemm_f16_common.h"

namespace dml {
namespace gemm16 {
namespace {

__device__ const half8 g_wide_zeros = {0, 0, 0, 0, 0, 0, 0, 0};   // what transfers past the end of K read

// T: 16 x 16 blocks of a wavefront in either direction; the four of a workgroup make a tile of 32 T x 32 T. AHEAD: steps that are
// on their way or in LDS beside the one that is multiplied; so many stages for A, one more for B.
template <int T> struct WideShape {
    static constexpr int kTile = 32 * T;
    static constexpr int kOperand = kTile * kRowBytes;   // bytes of one operand's tile
    static constexpr int kAhead = T == 8 ? 2 : 4;
    static constexpr int kLds = (2 * kAhead + 1) * kOperand;
};

template <bool FIRST>   // the first of a tile's products starts the sum
__device__ __forceinline__ void mfma_16x16x32(floatx4& acc, half8 b, half8 a) {
    if constexpr (FIRST) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc) : "v"(b), "v"(a));
    else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
}

// Four columns each of two neighbouring blocks: eight consecutive columns of the result. Behind the wait that follows the last
// MFMA; assembly, because the compiler copies all 256 accumulators to vector registers at once otherwise.
__device__ __forceinline__ void read_eight(const floatx4& a, const floatx4& b, float (&x)[8]) {
    asm volatile("v_accvgpr_read_b32 %0, %8\n\tv_accvgpr_read_b32 %1, %9\n\tv_accvgpr_read_b32 %2, %10\n\t"
                 "v_accvgpr_read_b32 %3, %11\n\tv_accvgpr_read_b32 %4, %12\n\tv_accvgpr_read_b32 %5, %13\n\t"
                 "v_accvgpr_read_b32 %6, %14\n\tv_accvgpr_read_b32 %7, %15"
                 : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7])
                 : "a"(a[0]), "a"(a[1]), "a"(a[2]), "a"(a[3]), "a"(b[0]), "a"(b[1]), "a"(b[2]), "a"(b[3]));
}

// Lanes l and l ^ 8 trade 16 bytes: p of the lanes 8 .. 15 of every sixteen against q of the lanes 0 .. 7.
__device__ __forceinline__ void trade(u32x4& p, u32x4& q) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t a = p[e], b = q[e];
        p[e] = __builtin_amdgcn_update_dpp(a, b, 0x128 /* row_ror:8 */, 0xf, 0xc, false);
        q[e] = __builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false);
    }
}

template <int T, int KIND, bool B> struct WideOperand;

// Where row r of a tile lies in LDS, or r itself for A. B's 16 x 16 blocks 2 p and 2 p + 1 take turns at four columns each of
// the 32 columns from 32 p on, so that a lane's four columns of both are eight consecutive ones.
__device__ __forceinline__ int b_row(int pos) {   // position j * 16 + 4 g + e -> 32 (j / 2) + 8 g + 4 (j % 2) + e
    return (pos & ~31) | (pos >> 2 & 3) << 3 | (pos >> 4 & 1) << 2 | (pos & 3);
}

template <int T, bool B> struct WideOperand<T, 0, B> {   // K contiguous
    int vo[T];          // byte offset of this lane's piece in transfer i of a step, from the tile's first row
    uint32_t faddr[2];  // this lane's fragment of block 0, either half of a step (stage 0)
    __device__ __forceinline__ void offsets(int64_t s_row, int64_t, int rows_left, int wave, int lane) {
        const int r0 = wave * 8 + (lane >> 3);
        const int c = (lane & 7) ^ swz16(r0);
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const int r = i * 32 + r0;
            vo[i] = (int)((min(B ? b_row(r) : r, rows_left - 1) * s_row + c * 8) * 2);
        }
    }
    __device__ __forceinline__ void fragments(uint32_t tile0, int row0, int lane) {
        const int r = row0 + (lane & 15);
#pragma unroll
        for (int s = 0; s < 2; ++s) faddr[s] = tile0 + r * kRowBytes + (((s * 4 + (lane >> 4)) ^ swz16(r)) << 4);
    }
    static __device__ __forceinline__ int64_t row_step(int64_t s_row) { return s_row; }
    // bytes from the tile's first element to the end of its last row
    static __device__ __forceinline__ uint32_t extent(int64_t s_row, int64_t, int rows_left, int k) {
        return (uint32_t)(((min(rows_left, 32 * T) - 1) * s_row + k) * 2);
    }
    static __device__ __forceinline__ uint32_t k_offset(int64_t, int step) { return (uint32_t)step * kRowBytes; }
    // transfer I of a step of which only `left` < 64 k exist (a multiple of 8: so is K of such an operand)
    template <int I>
    __device__ __forceinline__ void send_tail(const _Float16* tile, int64_t, int step, int left, char* dst, int wave, int lane) const {
        const char* p = reinterpret_cast<const char*>(tile) + k_offset(0, step) + (uint32_t)vo[I];
        const int kl = ((lane & 7) ^ swz16(wave * 8 + (lane >> 3))) * 8;
        lds_dma16(kl < left ? reinterpret_cast<const _Float16*>(p) : reinterpret_cast<const _Float16*>(&g_wide_zeros), dst);
    }
    template <int S, int U>
    __device__ __forceinline__ half8 fragment(uint32_t stage) const {
        return lds_read_b128<U * 16 * kRowBytes>(faddr[S] + stage);
    }
};

template <int T, bool B> struct WideOperand<T, 1, B> {   // rows contiguous
    static constexpr int P = 64 * T;          // bytes of a K row
    static constexpr int KPT = 4 * 1024 / P;  // K rows of the four wavefronts' transfers of one number
    int vo[T];
    uint32_t faddr[T];  // this lane's first transpose read of every 16-row block (stage 0)
    static __device__ __forceinline__ int k_of(int i, int wave, int lane) { return i * KPT + wave * (KPT / 4) + lane / (4 * T); }
    __device__ __forceinline__ void offsets(int64_t, int64_t s_k, int rows_left, int wave, int lane) {
        const int k0 = k_of(0, wave, lane);
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const int k = i * KPT + k0;
            const int c = (lane & (4 * T - 1)) ^ ((k & 3) << 2) ^ ((k >> 3 & 1) << 1);
            vo[i] = (int)((k * s_k + min(c * 8, rows_left - 8)) * 2);
        }
    }
    __device__ __forceinline__ void fragments(uint32_t tile0, int row0, int lane) {
        const int s = lane & 15, grp = lane >> 4;
        const int k = grp * 8 + (s >> 2);
#pragma unroll
        for (int u = 0; u < T; ++u) {
            const int row = row0 + (B ? b_row(u * 16 + 4 * (s & 3)) : u * 16 + 4 * (s & 3));
            faddr[u] = tile0 + k * P + (((row >> 3) ^ ((k & 3) << 2) ^ ((grp & 1) << 1)) << 4) + (row & 7) * 2;
        }
    }
    static __device__ __forceinline__ int64_t row_step(int64_t) { return 1; }
    static __device__ __forceinline__ uint32_t extent(int64_t, int64_t s_k, int rows_left, int k) {
        return (uint32_t)(((k - 1) * s_k + min(rows_left, 32 * T)) * 2);
    }
    static __device__ __forceinline__ uint32_t k_offset(int64_t s_k, int step) { return (uint32_t)(step * BK * s_k * 2); }
    // transfer I of a step of which only `left` < 64 k exist
    template <int I>
    __device__ __forceinline__ void send_tail(const _Float16* tile, int64_t s_k, int step, int left, char* dst, int wave, int lane) const {
        const char* p = reinterpret_cast<const char*>(tile) + k_offset(s_k, step) + (uint32_t)vo[I];
        lds_dma16(k_of(I, wave, lane) < left ? reinterpret_cast<const _Float16*>(p) : reinterpret_cast<const _Float16*>(&g_wide_zeros), dst);
    }
    template <int S, int U>
    __device__ __forceinline__ half8 fragment(uint32_t stage) const {
        const uint32_t a = faddr[U] + stage;
        const half4v lo = lds_read_tr16_b64<S * 32 * P>(a);
        const half4v hi = lds_read_tr16_b64<S * 32 * P + 4 * P>(a);
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
};

__device__ __forceinline__ void* uniform(const void* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<void*>((uint64_t)hi << 32 | lo);
}

// Where a tile is and what its operands' transfers read: all of it uniform.
struct WideTile {
    int m0, n0, z0, z1;
    int64_t aoff, boff, coff;   // element offsets of the batch entry
};

template <int T>
__device__ __forceinline__ WideTile wide_tile(const GemmArgs& g, uint32_t bid) {
    {   // contiguous runs of tiles per XCD; workgroups are dealt to the XCDs in turn
        const uint32_t total = (uint32_t)g.total_blocks;
        const uint32_t xcd = bid % kXcds, idx = bid / kXcds;
        const uint32_t base = total / kXcds, rem = total % kXcds;
        bid = xcd * base + (xcd < rem ? xcd : rem) + idx;
    }
    const uint32_t tiles = (uint32_t)(g.tiles_m * g.tiles_n);
    uint32_t batch = 0, tile = bid;
    if (bid >= tiles) {
        batch = bid / tiles;
        tile = bid - batch * tiles;
    }
    // groups of eight tile rows, column by column (gemm_f16_pipe.h)
    constexpr uint32_t kGroupM = 8;
    const uint32_t per_group = kGroupM * (uint32_t)g.tiles_n;
    const uint32_t group = tile / per_group, in_group = tile - group * per_group;
    const uint32_t rows_here = min((uint32_t)g.tiles_m - group * kGroupM, kGroupM);
    const uint32_t tn = in_group / rows_here;
    WideTile t;
    t.m0 = (int)(group * kGroupM + (in_group - tn * rows_here)) * WideShape<T>::kTile;
    t.n0 = (int)tn * WideShape<T>::kTile;
    int z2 = 0;
    t.z0 = t.z1 = 0;
    if (batch != 0) {
        const uint32_t b2 = (uint32_t)g.batch2, b1 = (uint32_t)g.batch1;
        const uint32_t q = batch / b2;
        z2 = (int)(batch - q * b2);
        t.z0 = (int)(q / b1);
        t.z1 = (int)(q - (uint32_t)t.z0 * b1);
    }
    t.aoff = t.z0 * g.sab[0] + t.z1 * g.sab[1] + z2 * g.sab[2];
    t.boff = t.z0 * g.sbb[0] + t.z1 * g.sbb[1] + z2 * g.sbb[2];
    t.coff = t.z0 * g.scb[0] + t.z1 * g.scb[1] + z2 * g.scb[2];
    return t;
}

// alpha, biases and residual as in store_strip (gemm_f16_common.h), for eight consecutive columns of one row
template <typename OutT, int EPI>
__device__ __forceinline__ void wide_result(const GemmArgs& g, bool residual, typename OutVec<OutT>::type rv, float bm,
                                            const float (&bias)[8], float (&v)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = v[e] * g.alpha + bias[e];
    if constexpr (EPI == EPI_GENERAL) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += bm;
        if (residual) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += (float)rv[e];
        }
    }
}

// 16 bytes of the result. A workgroup's last fp16 tile goes through the L2 as it is written (global_store_b128_through). The
// tiles before it stay in the L2, which takes them faster than the memory behind it and writes them back under the next
// tile's loop.
template <typename OutT>
__device__ __forceinline__ void wide_store(OutT* p, u32x4 v, bool through) {
    if (sizeof(OutT) == 2 && through) global_store_b128_through(p, __builtin_bit_cast(half8, v));
    else *reinterpret_cast<u32x4*>(p) = v;
}

// The wavefront's 128 x 128 tile in strips of 16 rows and 32 columns (fp32) or 64 (fp16): lane l has columns 8 (l / 16) .. + 7
// of every 32 of row l % 16. Lanes l and l ^ 8 trade half of a strip, so that a store instruction writes 128 bytes each of
// eight rows: 64 bytes each of sixteen rows take twice as long (12.2 against 6.1 us for a 4096 x 4096 result).
template <int T, typename OutT, int EPI>
__device__ __forceinline__ void wide_epilogue(const GemmArgs& g, void* c_ptr, const void* res_ptr, const void* bias_ptr,
                                              const floatx4 (&acc)[T][T], int mb, int nb, int64_t coff, int lane, bool through) {
    typedef typename OutVec<OutT>::type ovec;
    constexpr bool GENERAL = EPI == EPI_GENERAL;
    constexpr bool HALF = sizeof(OutT) == 2;
    OutT* C = reinterpret_cast<OutT*>(c_ptr);
    const OutT* R = reinterpret_cast<const OutT*>(res_ptr);
    const int col = (lane >> 4) * 8, row = lane & 15;
    float bias[T / 2][8];
#pragma unroll
    for (int p = 0; p < T / 2; ++p) {
        const int n = min(nb + p * 32 + col, g.n - 8);
        if (!bias_ptr || g.bias_m) {
#pragma unroll
            for (int e = 0; e < 8; ++e) bias[p][e] = 0.f;
        } else if (g.bias_f32) {
            const floatx4 b0 = *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(bias_ptr) + n);
            const floatx4 b1 = *reinterpret_cast<const floatx4*>(reinterpret_cast<const float*>(bias_ptr) + n + 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) { bias[p][e] = b0[e]; bias[p][e + 4] = b1[e]; }
        } else {
            const half8 b = *reinterpret_cast<const half8*>(reinterpret_cast<const _Float16*>(bias_ptr) + n);
#pragma unroll
            for (int e = 0; e < 8; ++e) bias[p][e] = (float)b[e];
        }
    }
    // what has to be loaded (general variant only): four strips of 16 rows ahead of the stores of the first
    constexpr int AHEAD = GENERAL ? (HALF ? 4 : 2) : 1;
    static_for<0, T / AHEAD>([&](auto hc) {
        constexpr int i0 = decltype(hc)::value * AHEAD;
        ovec rv[AHEAD][T / 2];
        float bm[AHEAD];
        if constexpr (GENERAL) {
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) {
                const int m = min(mb + (i0 + i) * 16 + row, g.m - 1);
                bm[i] = 0.f;
                if (bias_ptr && g.bias_m)
                    bm[i] = g.bias_f32 ? reinterpret_cast<const float*>(bias_ptr)[m]
                                       : (float)reinterpret_cast<const _Float16*>(bias_ptr)[m];
#pragma unroll
                for (int p = 0; p < T / 2; ++p)
                    if (R) rv[i][p] = *reinterpret_cast<const ovec*>(R + coff + (int64_t)m * g.scm + min(nb + p * 32 + col, g.n - 8));
            }
        }
        static_for<0, AHEAD>([&](auto ic) {
            constexpr int ii = decltype(ic)::value, i = i0 + ii;
            const int m = mb + i * 16 + (row & 7);
            static_for<0, HALF ? T / 4 : T / 2>([&](auto pc) {
                constexpr int p = decltype(pc)::value * (HALF ? 2 : 1);
                u32x4 lo, hi;
                int n;
                if constexpr (HALF) {   // lanes 0 .. 7 end up with these 32 columns of two rows, lanes 8 .. 15 with the next 32
                    float x[8], y[8];
                    read_eight(acc[i][2 * p], acc[i][2 * p + 1], x);
                    read_eight(acc[i][2 * p + 2], acc[i][2 * p + 3], y);
                    wide_result<OutT, EPI>(g, R != nullptr, rv[ii][p], bm[ii], bias[p], x);
                    wide_result<OutT, EPI>(g, R != nullptr, rv[ii][p + 1], bm[ii], bias[p + 1], y);
                    half8 hx, hy;
#pragma unroll
                    for (int e = 0; e < 8; ++e) { hx[e] = (_Float16)x[e]; hy[e] = (_Float16)y[e]; }
                    lo = __builtin_bit_cast(u32x4, hx);
                    hi = __builtin_bit_cast(u32x4, hy);
                    n = nb + p * 32 + col + (row >> 3) * 32;
                } else {                // ... with the first four of their eight columns, with the others
                    float x[8];
                    read_eight(acc[i][2 * p], acc[i][2 * p + 1], x);
                    wide_result<OutT, EPI>(g, R != nullptr, rv[ii][p], bm[ii], bias[p], x);
#pragma unroll
                    for (int e = 0; e < 4; ++e) { lo[e] = __builtin_bit_cast(uint32_t, x[e]); hi[e] = __builtin_bit_cast(uint32_t, x[e + 4]); }
                    n = nb + p * 32 + col + (row >> 3) * 4;
                }
                trade(lo, hi);
                OutT* const c = C + coff + (int64_t)m * g.scm + n;
                if (m < g.m && n < g.n) wide_store(c, lo, through);
                if (m + 8 < g.m && n < g.n) wide_store(c + 8 * g.scm, hi, through);
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    });
}

// SLICED: the inner batch index z1 counts g.batch1 slices of K (its operand strides are 0); g.asum, if any, receives the partial
// row sums [z0][z1][tile column][2][m] in fp32.
template <int T, int AKIND, int BKIND, int EPI, bool KSUM, bool SLICED = false>
__global__ __launch_bounds__(kThreads) void gemm_f16_wide_kernel(const _Float16* a_ptr, const _Float16* b_ptr, void* c_ptr,
                                                                 const void* bias_ptr, const void* res_ptr, const GemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)   // buffer descriptors exist on the device only
    constexpr int NM = T * T, TILE = WideShape<T>::kTile, OPERAND = WideShape<T>::kOperand, AHEAD = WideShape<T>::kAhead;
    constexpr int WT = TILE / 2;       // rows and columns of a wavefront
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int wm = wave >> 1, wn = wave & 1;
    if (g.trace && threadIdx.x == 0) g.trace[4 * (size_t)blockIdx.x] = wall_clock64();

    WideOperand<T, AKIND, false> oa;
    WideOperand<T, BKIND, true> ob;
    const uint32_t lds0 = lds_addr(lds);
    oa.fragments(lds0, wm * WT, lane);
    ob.fragments(lds0 + AHEAD * OPERAND, wn * WT, lane);

    static_assert(!SLICED || (AKIND == 1 && EPI == EPI_PLAIN && !KSUM), "slices are for weight gradients");
    const int nkg = SLICED ? (g.k + BK - 1) / BK : g.k / BK;   // steps of one operand pair
    auto slice_begin = [&](int z1) { return (int)((uint32_t)nkg * (uint32_t)z1 / (uint32_t)g.batch1); };
    uint32_t bid = blockIdx.x;
    const uint32_t total = (uint32_t)g.total_blocks;

    // ---- what the transfers read: two steps ahead of the MFMAs, past the end of a tile the first steps of the next one
    __amdgpu_buffer_rsrc_t ra, rb;
    const _Float16 *tile_a = nullptr, *tile_b = nullptr;   // where they begin, for the ragged step
    uint32_t fbid = bid;   // the tile they belong to, which is ahead of the one that is multiplied
    int fk = 0, fend = nkg, fgrp = 0, rows_a = 0, rows_b = 0;
    auto point_at = [&](uint32_t at) {
        const WideTile ft = wide_tile<T>(g, at);
        fk = 0;
        if constexpr (SLICED) {
            fk = slice_begin(ft.z1);
            fend = slice_begin(ft.z1 + 1);
        }
        const _Float16 *a = a_ptr, *b = b_ptr;
        if constexpr (KSUM) {
            // constant indices: the table stays in the kernel-argument segment
            a = fgrp == 0 ? g.ga[0] : fgrp == 1 ? g.ga[1] : fgrp == 2 ? g.ga[2] : g.ga[3];
            b = fgrp == 0 ? g.gb[0] : fgrp == 1 ? g.gb[1] : fgrp == 2 ? g.gb[2] : g.gb[3];
        } else if (g.groups) {
            a = g.ga[ft.z0];
            b = g.gb[ft.z0];
        }
        a += ft.aoff + ft.m0 * WideOperand<T, AKIND, false>::row_step(g.sam);
        b += ft.boff + ft.n0 * WideOperand<T, BKIND, true>::row_step(g.sbn);
        if constexpr (SLICED) {
            tile_a = a;
            tile_b = b;
        }
        const int la = g.m - ft.m0, lb = g.n - ft.n0;
        // rows past the end of an operand read its last row; the descriptor ends where the operand does
        ra = __builtin_amdgcn_make_buffer_rsrc(uniform(a), 0, (int)WideOperand<T, AKIND, false>::extent(g.sam, g.sak, la, g.k), 0x00020000);
        rb = __builtin_amdgcn_make_buffer_rsrc(uniform(b), 0, (int)WideOperand<T, BKIND, true>::extent(g.sbn, g.sbk, lb, g.k), 0x00020000);
        if (min(la, TILE) != rows_a) {
            rows_a = min(la, TILE);
            oa.offsets(g.sam, g.sak, rows_a, wave, lane);
        }
        if (min(lb, TILE) != rows_b) {
            rows_b = min(lb, TILE);
            ob.offsets(g.sbn, g.sbk, rows_b, wave, lane);
        }
    };
    point_at(fbid);
    auto send_a = [&](auto ic, int stage) {
        constexpr int i = decltype(ic)::value;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            ra, (__attribute__((address_space(3))) void*)(lds + stage * OPERAND + (i * 4 + wave) * 1024), 16, oa.vo[i],
            (int)WideOperand<T, AKIND, false>::k_offset(g.sak, fk), 0, 0);
    };
    auto send_b = [&](auto ic, int stage) {
        constexpr int i = decltype(ic)::value;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rb, (__attribute__((address_space(3))) void*)(lds + (AHEAD + stage) * OPERAND + (i * 4 + wave) * 1024), 16, ob.vo[i],
            (int)WideOperand<T, BKIND, true>::k_offset(g.sbk, fk), 0, 0);
    };
    // the next step of this tile, or the first of the next one (of the last one: nothing is sent any more)
    auto advance = [&]() {
        if (++fk != fend) return;
        if (KSUM && ++fgrp != g.groups) {
            point_at(fbid);   // a pair of few steps ends while the tile before is still being multiplied
            return;
        }
        fgrp = 0;
        fbid += gridDim.x;
        if (fbid < total) point_at(fbid);
    };

    for (int s = 0; s < AHEAD; ++s) {
        static_for<0, T>([&](auto i) { send_b(i, s); });
        static_for<0, T>([&](auto i) { send_a(i, s); });
        advance();
    }
    wait_vm_lgkm0<(AHEAD - 1) * 2 * T>();
    __builtin_amdgcn_s_barrier();
    if (g.trace && threadIdx.x == 0) g.trace[4 * (size_t)blockIdx.x + 1] = wall_clock64();

    constexpr int kReadEvery = T == 8 ? 2 : 1;   // MFMAs per fragment read
    half8 af[2][T], bf[2][T];   // fragments of the first and the second 32 k of a step
    auto read = [&](auto uc, auto sc, uint32_t a_stage, uint32_t b_stage) {
        constexpr int u = decltype(uc)::value, s = decltype(sc)::value;
        if constexpr (u < T) bf[s][u] = ob.template fragment<s, u>(b_stage);
        else af[s][u - T] = oa.template fragment<s, u - T>(a_stage);
    };
    static_for<0, 2 * T>([&](auto u) { read(u, std::integral_constant<int, 0>{}, 0u, 0u); });

    floatx4 acc[T][T];
    int as = 0, bs = 0;   // stages of the step that is multiplied
    float row_sum[SLICED ? T : 1];   // row lane % 16 of every block, the k of this lane's fragments
    int sum_in = -1;                 // steps until this workgroup sums fragments again
    // FIRST: of a tile. LEFT: steps that follow, AHEAD for more; with as many the step that far ahead is sent, with one the next
    // step's first fragments are read. TAIL: what is sent is the ragged last step of K.
    auto step = [&](auto first_c, auto left_c, auto tail_c) {
        constexpr bool FIRST = decltype(first_c)::value, TAIL = decltype(tail_c)::value;
        constexpr int LEFT = decltype(left_c)::value;
        constexpr bool FILL = LEFT == AHEAD, MORE = LEFT > 0;
        const int an = as == AHEAD - 1 ? 0 : as + 1, bn = bs == AHEAD ? 0 : bs + 1, bfill = bs == 0 ? AHEAD : bs - 1;
        static_for<0, 2>([&](auto sc) {
            constexpr int s = decltype(sc)::value;
            if constexpr (s == 1 && MORE) {
                // this wavefront's transfers of the next step have landed (loads complete in order; those of the steps behind
                // it, B's half of a step sent so far among them, may be on their way, whatever stores are outstanding) and its
                // last fragments of this step are in registers; behind the barrier, everybody's
                wait_vm_lgkm0<FILL ? (AHEAD - 2) * 2 * T + T : (LEFT - 1) * 2 * T>();
                __builtin_amdgcn_s_barrier();
            } else {
                wait_lgkm<0>();
            }
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, NM>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                constexpr int i = m / T, j = (i & 1) ? T - 1 - m % T : m % T;
                mfma_16x16x32<FIRST && s == 0>(acc[i][j], bf[s][j], af[s][i]);
                if constexpr (m % kReadEvery == 0 && m / kReadEvery < 2 * T) {
                    if constexpr (s == 0) read(std::integral_constant<int, m / kReadEvery>{}, std::integral_constant<int, 1>{}, as * OPERAND, bs * OPERAND);
                    else if constexpr (MORE) read(std::integral_constant<int, m / kReadEvery>{}, std::integral_constant<int, 0>{}, an * OPERAND, bn * OPERAND);
                }
                if constexpr (FILL && TAIL && m % T == 1) {
                    constexpr int d = m / T;
                    if constexpr (s == 0) ob.template send_tail<d>(tile_b, g.sbk, fk, g.k - fk * BK, lds + (AHEAD + bfill) * OPERAND + (d * 4 + wave) * 1024, wave, lane);
                    else oa.template send_tail<d>(tile_a, g.sak, fk, g.k - fk * BK, lds + as * OPERAND + (d * 4 + wave) * 1024, wave, lane);
                } else if constexpr (FILL && m % T == 1) {
                    if constexpr (s == 0) send_b(std::integral_constant<int, m / T>{}, bfill);
                    else send_a(std::integral_constant<int, m / T>{}, as);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            // the two wavefronts that share these rows of A take one half of the step each
            if constexpr (SLICED) {
                if (sum_in == 0 && wn == s) {
                    const half2v one2 = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
                    for (int i = 0; i < T; ++i)
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            const half2v p = {af[s][i][e], af[s][i][e + 1]};
                            row_sum[i] = __builtin_amdgcn_fdot2(p, one2, row_sum[i], false);
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        if constexpr (SLICED) sum_in = sum_in == 0 ? g.tiles_n - 1 : sum_in - 1;
        if constexpr (FILL) advance();
        as = an;
        bs = bn;
    };

    using yes = std::true_type;
    using no = std::false_type;
    using full = std::integral_constant<int, AHEAD>;
    for (;;) {
        const bool last = bid + gridDim.x >= total;
        const WideTile t = wide_tile<T>(g, bid);
        int nk = KSUM ? nkg * g.groups : nkg;
        if constexpr (SLICED) {
            nk = slice_begin(t.z1 + 1) - slice_begin(t.z1);
            sum_in = g.asum ? t.n0 / TILE : -1;
#pragma unroll
            for (int i = 0; i < T; ++i) row_sum[i] = 0.f;
        }
        const int fills = last ? nk - AHEAD : nk;
        step(yes{}, full{}, no{});
        if constexpr (SLICED) {
            // the last slice's last step may be ragged: it is sent AHEAD steps before (the host passes a step more then)
            const int tail = g.k % BK != 0 && t.z1 + 1 == g.batch1 ? nk - 1 - AHEAD : -1;
            int kt = 1;
            for (; kt < fills && kt != tail; ++kt) step(no{}, full{}, no{});
            if (kt == tail) {
                step(no{}, full{}, yes{});
                for (++kt; kt < fills; ++kt) step(no{}, full{}, no{});
            }
        } else {
            for (int kt = 1; kt < fills; ++kt) step(no{}, full{}, no{});
        }
        if (last) static_for<1, AHEAD + 1>([&](auto lc) { step(no{}, std::integral_constant<int, AHEAD - decltype(lc)::value>{}, no{}); });
        // an accumulator is read no earlier than 18 wait states behind the last MFMA (the assembly hides them from the compiler),
        // and the next tile's first fragments are in their registers before the epilogue may use others around them
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15\n\ts_nop 3" ::: "memory");
        if (last && g.trace && threadIdx.x == 0) g.trace[4 * (size_t)blockIdx.x + 2] = wall_clock64();
        void* c = c_ptr;
        const void* bias = bias_ptr;
        if (!KSUM && g.groups) {
            c = g.gc[t.z0];
            bias = g.gbias[t.z0];
        }
        const int mb = t.m0 + wm * WT, nb = t.n0 + wn * WT;
        if (g.out_f32) wide_epilogue<T, float, EPI>(g, c, res_ptr, bias, acc, mb, nb, t.coff, lane, last);
        else wide_epilogue<T, _Float16, EPI>(g, c, res_ptr, bias, acc, mb, nb, t.coff, lane, last);
        if constexpr (SLICED) {
            if (g.asum) {
                float* const sums = reinterpret_cast<float*>(g.asum) +
                                    ((((int64_t)t.z0 * g.batch1 + t.z1) * g.tiles_n + t.n0 / TILE) * 2 + wn) * g.m;
#pragma unroll
                for (int i = 0; i < T; ++i) {
                    float v = row_sum[i];
                    v += __shfl_xor(v, 16);
                    v += __shfl_xor(v, 32);
                    const int m = mb + i * 16 + lane;
                    if (lane < 16 && m < g.m) sums[m] = v;
                }
            }
        }
        if (last) break;
        bid += gridDim.x;
    }
    if (g.trace && threadIdx.x == 0) {
        wait_vm_lgkm0<0>();   // this wavefront's stores have been accepted
        g.trace[4 * (size_t)blockIdx.x + 3] = wall_clock64();
    }
#endif
}

// ---------------------------------------------------------------- host side
template <int T, int AKIND, int BKIND, int EPI, bool KSUM, bool SLICED = false>
int launch_shape(const GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* residual,
                 hipStream_t st) {
    auto kern = gemm_f16_wide_kernel<T, AKIND, BKIND, EPI, KSUM, SLICED>;
    constexpr int lds = WideShape<T>::kLds;
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
        set_error("gemm_f16: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
        return (int)e;
    }
    const unsigned grid = (unsigned)(g.total_blocks < kCus ? g.total_blocks : kCus);
    hipLaunchKernelGGL(kern, grid, kThreads, lds, st, a, b, c, bias, residual, g);
    return launch_status("gemm_f16(wide)");
}

inline int wide_unsupported(int ak, int bk) {
    set_error("gemm_f16: no kernel with tiles that stay for operand kinds %d/%d", ak, bk);
    return DMLHIP_ERR_UNSUPPORTED;
}

#define DML_WIDE_TILES(T)                                                                                          \
    constexpr int tile = WideShape<T>::kTile;                                                                      \
    g.tiles_m = (g.m + tile - 1) / tile;                                                                           \
    g.tiles_n = (g.n + tile - 1) / tile;                                                                           \
    const long long total = (long long)g.tiles_m * g.tiles_n * batch;                                              \
    DML_REQUIRE(total <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f16: %lld workgroups exceed the grid limit", total); \
    g.total_blocks = total;                                                                                        \
    const int ek = epilogue_kind(g, bias, residual, nullptr);
#define DML_WIDE_CASE(T, AK, BKD, EPI, KSUM)                    \
    if (ak == AK && bk == BKD && ek == EPI && !!g.ksum == KSUM) \
        return launch_shape<T, AK, BKD, EPI, KSUM>(g, a, b, c, bias, residual, st);
#define DML_WIDE_CASES(T, AK, BKD)                                                                  \
    DML_WIDE_CASE(T, AK, BKD, EPI_PLAIN, false) DML_WIDE_CASE(T, AK, BKD, EPI_GENERAL, false) \
    DML_WIDE_CASE(T, AK, BKD, EPI_PLAIN, true) DML_WIDE_CASE(T, AK, BKD, EPI_GENERAL, true)

// Adds up what SLICED left: blocks of 1024 results each, behind them (asum) blocks of 64 row sums; the group in blockIdx.y.
// Reads of 4 bytes per result and slice and the result's own: 3.3 TB/s behind the product, 80 MB in 24 us.
struct WideSumArgs {
    const float* part;        // [groups][slices][count]
    const float* row_part;    // [groups][row_parts][m]
    int slices, row_parts, m, out_f32, asum_f32;
    int64_t count;
    float alpha;
    void* out[DMLHIP_GROUP_MAX];
    void* asum[DMLHIP_GROUP_MAX];
};

__global__ __launch_bounds__(256) void wide_sum_kernel(const WideSumArgs g, int blocks) {
    const int z = blockIdx.y;
    if ((int)blockIdx.x < blocks) {
        const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
        if (i >= g.count) return;
        const float* p = g.part + (int64_t)z * g.slices * g.count + i;
        floatx4 acc = *reinterpret_cast<const floatx4*>(p);
#pragma unroll 4
        for (int s = 1; s < g.slices; ++s) acc += *reinterpret_cast<const floatx4*>(p + (int64_t)s * g.count);
        acc *= g.alpha;
        if (g.out_f32) {
            *reinterpret_cast<floatx4*>(reinterpret_cast<float*>(g.out[z]) + i) = acc;
        } else {
            const half4v h = {(_Float16)acc[0], (_Float16)acc[1], (_Float16)acc[2], (_Float16)acc[3]};
            *reinterpret_cast<half4v*>(reinterpret_cast<_Float16*>(g.out[z]) + i) = h;
        }
        return;
    }
    __shared__ float share[256];
    const int row = ((int)blockIdx.x - blocks) * 64 + (threadIdx.x & 63);
    float v = 0.f;
    if (row < g.m) {
        const float* p = g.row_part + (int64_t)z * g.row_parts * g.m + row;
#pragma unroll 4
        for (int q = threadIdx.x >> 6; q < g.row_parts; q += 4) v += p[(int64_t)q * g.m];
    }
    share[threadIdx.x] = v;
    __syncthreads();
    if (threadIdx.x < 64 && row < g.m) {
        v = (share[threadIdx.x] + share[threadIdx.x + 64]) + (share[threadIdx.x + 128] + share[threadIdx.x + 192]);
        if (g.asum_f32) reinterpret_cast<float*>(g.asum[z])[row] = v;
        else reinterpret_cast<_Float16*>(g.asum[z])[row] = (_Float16)v;
    }
}

}  // namespace
}  // namespace gemm16
}  // namespace dml
