// fp16 x fp16 -> fp32-accumulate strided batched GEMM on the gfx950 matrix cores
// (v_mfma_f32_32x32x16_f16), the kernel behind MatMul / Einsum / Gemm and their backward
// contractions.
//
// Tiling: a workgroup of 4 wavefronts owns a BM x BN tile of C and walks K in steps of 64.
// Each K step stages an A tile [BM][64] and a B tile [BN][64] (both K-contiguous, 128 bytes per
// row) in LDS, double-buffered, so one barrier per step. Global loads for step t+1 are issued
// before the MFMAs of step t and written to the other LDS buffer afterwards.
//
// LDS layout: rows are split into eight 16-byte chunks; chunk c of row r is stored at chunk slot
// c ^ ((r ^ (r >> 3)) & 7). A fragment read (lane -> row l%32, chunk 2*kk + l/32) then touches
// eight distinct slots per eight consecutive rows, and so do both kinds of tile stores.
//
// Operand layout: each operand may be K-contiguous (stride_k == 1; 128-bit loads straight to LDS)
// or row-contiguous (stride_m/n == 1, i.e. the transposed storage). The latter is transposed in
// registers on the way to LDS: a thread loads eight K-rows of RU adjacent rows and re-packs them
// into RU chunks of eight K values, so no separate transpose kernel or HBM round trip is needed.
#include "gemm_f16_common.h"

#include <atomic>

namespace dml {
using namespace gemm16;
namespace {

// ---------------------------------------------------------------- global -> registers
// The loaders are branch-free in the steady state. Rows past the end of the operand are clamped to
// the last valid row (they only feed rows/columns of C that are never stored); K past the end is
// zero-filled, and only the last K step takes that path. Offsets are 32-bit element offsets from
// the operand's batch base (the host falls back to the generic loader when they would not fit).

// K-contiguous operand (k % 8 == 0): thread t loads chunks q = t + i*256 of the [R][64] tile.
// Loads never branch: a chunk past the end of K is fetched from the last valid chunk instead and
// replaced by zeros when it is written to LDS.
template <int R>
struct LoaderKC {
    static constexpr int N = R * 8 / kThreads;
    u32x4 v[N];
    int off[N];
    int c8;       // first k of this thread's chunk inside a K step
    int k_valid;  // k of the tile held in v[] minus its k0 (chunks with c8 >= k_valid are zero)
    __device__ __forceinline__ void init(int64_t s_row, int64_t, int row0, int rows) {
        c8 = (threadIdx.x & 7) * 8;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = threadIdx.x + i * kThreads;
            const int r = min(row0 + (q >> 3), rows - 1);
            off[i] = (int)(r * s_row);
        }
    }
    __device__ __forceinline__ void load(const _Float16* base, int64_t, int k0, int k) {
        k_valid = k - k0;
        const int kc = min(k0 + c8, k - 8);
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = *reinterpret_cast<const u32x4*>(base + off[i] + kc);
    }
    __device__ __forceinline__ void store(char* tile) const {
        const bool ok = c8 < k_valid;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = threadIdx.x + i * kThreads;
            const int r = q >> 3, c = q & 7;
            const u32x4 z = {0u, 0u, 0u, 0u};
            *reinterpret_cast<u32x4*>(tile + r * kRowBytes + ((c ^ swz(r)) << 4)) = ok ? v[i] : z;
        }
    }
};

// K-contiguous operand with k % 64 == 0, loaded straight into LDS (global_load_lds, 16 bytes per
// lane): no staging registers and no LDS store instructions. One wave instruction fills 1 KiB =
// eight tile rows; lane l lands at (row l/8, chunk slot l%8) of that group, so it fetches the
// global chunk that the swizzle maps to this slot.
template <int R>
struct LoaderKCDirect {
    static constexpr int N = R / 32;  // instructions per wavefront per tile
    int off[N];
    int wave;
    __device__ __forceinline__ void init(int64_t s_row, int64_t, int row0, int rows) {
        const int lane = threadIdx.x & (kWave - 1);
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int r = (i * 4 + wave) * 8 + (lane >> 3);
            const int c = (lane & 7) ^ swz(r);
            off[i] = (int)(min(row0 + r, rows - 1) * s_row) + c * 8;
        }
    }
    __device__ __forceinline__ void issue(const _Float16* base, int k0, char* tile) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(base + off[i] + k0),
                (__attribute__((address_space(3))) void*)(tile + (i * 4 + wave) * 1024), 16, 0, 0);
        }
    }
    __device__ __forceinline__ void load(const _Float16*, int64_t, int, int) {}
    __device__ __forceinline__ void store(char*) const {}
};

// Row-contiguous operand (element (row, k) at k*s_k + row; rows % RU == 0): thread t owns K block
// kb = t/32 (eight K values) of the RU rows starting at (t%32)*RU and transposes them in registers.
// K rows past the end are fetched from row k-1 and zeroed on the way to LDS.
template <int R>
struct LoaderRC {
    static constexpr int RU = R / 32;  // 4 for R=128, 8 for R=256
    typedef _Float16 rowvec __attribute__((ext_vector_type(RU)));
    rowvec v[8];
    int off;
    int k_valid;
    __device__ __forceinline__ void init(int64_t, int64_t, int row0, int rows) {
        const int rg = threadIdx.x & 31;
        off = min(row0 + rg * RU, rows - RU);
    }
    __device__ __forceinline__ void load(const _Float16* base, int64_t s_k, int k0, int k) {
        const int kb8 = (threadIdx.x >> 5) * 8;
        k_valid = k - k0 - kb8;
        const _Float16* p = base + off;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int gk = min(k0 + kb8 + j, k - 1);
            v[j] = *reinterpret_cast<const rowvec*>(p + (int64_t)gk * s_k);
        }
    }
    __device__ __forceinline__ void store(char* tile) const {
        const int kb = threadIdx.x >> 5, rg = threadIdx.x & 31;
#pragma unroll
        for (int e = 0; e < RU; ++e) {
            half8 o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = j < k_valid ? v[j][e] : (_Float16)0;
            const int r = rg * RU + e;
            *reinterpret_cast<half8*>(tile + r * kRowBytes + ((kb ^ swz(r)) << 4)) = o;
        }
    }
};

// Any strides, any alignment: guarded element loads. Correct everywhere, fast nowhere.
template <int R>
struct LoaderGeneric {
    static constexpr int N = R * 8 / kThreads;
    half8 v[N];
    int64_t s_row_, s_k_;
    int row0_, rows_;
    __device__ __forceinline__ void init(int64_t s_row, int64_t s_k, int row0, int rows) {
        s_row_ = s_row; s_k_ = s_k; row0_ = row0; rows_ = rows;
    }
    __device__ __forceinline__ void load(const _Float16* base, int64_t, int k0, int k) {
#pragma unroll 1
        for (int i = 0; i < N; ++i) {
            const int q = threadIdx.x + i * kThreads;
            const int r = q >> 3, c = q & 7;
            const int gr = row0_ + r, gk = k0 + c * 8;
            half8 h = {};
            if (gr < rows_) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (gk + e < k) h[e] = base[(int64_t)gr * s_row_ + (int64_t)(gk + e) * s_k_];
            }
            v[i] = h;
        }
    }
    __device__ __forceinline__ void store(char* tile) const {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int q = threadIdx.x + i * kThreads;
            const int r = q >> 3, c = q & 7;
            *reinterpret_cast<half8*>(tile + r * kRowBytes + ((c ^ swz(r)) << 4)) = v[i];
        }
    }
};

template <int R, int MODE> struct LoaderSel;
template <int R> struct LoaderSel<R, 0> { using type = LoaderKC<R>; };
template <int R> struct LoaderSel<R, 1> { using type = LoaderRC<R>; };
template <int R> struct LoaderSel<R, 2> { using type = LoaderGeneric<R>; };
template <int R> struct LoaderSel<R, 3> { using type = LoaderKCDirect<R>; };

// ---------------------------------------------------------------- the kernel
// AMODE / BMODE: 0 = K-contiguous via registers, 1 = row-contiguous, 2 = generic strides,
// 3 = K-contiguous straight to LDS (k % 64 == 0).
template <int BM, int BN, int WM, int WN, int AMODE, int BMODE, bool ACT>
__global__ __launch_bounds__(kThreads) void gemm_f16_kernel(const _Float16* __restrict__ a_ptr,
                                                            const _Float16* __restrict__ b_ptr, void* c_ptr,
                                                            const void* bias_ptr, const void* res_ptr, void* pre_ptr,
                                                            const GemmArgs g) {
    static_assert((BM / WM) * (BN / WN) == kThreads / kWave, "four wavefronts per workgroup");
    constexpr int TM = WM / 32, TN = WN / 32;
    constexpr int A_BYTES = BM * kRowBytes, B_BYTES = BN * kRowBytes;
    extern __shared__ __attribute__((aligned(16))) char lds[];

    // ---- block -> (batch, tile): blocks are dealt round-robin to the eight XCDs, so give each
    // XCD a contiguous run of tiles (neighbouring tiles share operand panels in that XCD's L2).
    long long bid = blockIdx.x;
    {
        const long long total = g.total_blocks;
        const long long xcd = bid % kXcds, idx = bid / kXcds;
        const long long base = total / kXcds, rem = total % kXcds;
        bid = xcd * base + (xcd < rem ? xcd : rem) + idx;
    }
    const int tiles = g.tiles_m * g.tiles_n;
    const long long batch = bid / tiles;
    const int tile = (int)(bid % tiles);
    const int tm = tile / g.tiles_n, tn = tile % g.tiles_n;
    const int z2 = (int)(batch % g.batch2);
    const int z1 = (int)((batch / g.batch2) % g.batch1);
    const int z0 = (int)(batch / ((long long)g.batch2 * g.batch1));
    const _Float16* A = a_ptr + z0 * g.sab[0] + z1 * g.sab[1] + z2 * g.sab[2];
    const _Float16* B = b_ptr + z0 * g.sbb[0] + z1 * g.sbb[1] + z2 * g.sbb[2];
    const int64_t coff = z0 * g.scb[0] + z1 * g.scb[1] + z2 * g.scb[2];
    const int m0 = tm * BM, n0 = tn * BN;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int wm = wave / (BN / WN), wn = wave % (BN / WN);

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    typename LoaderSel<BM, AMODE>::type la;
    typename LoaderSel<BN, BMODE>::type lb;

    const int nk = (g.k + BK - 1) / BK;
    la.init(g.sam, g.sak, m0, g.m);
    lb.init(g.sbn, g.sbk, n0, g.n);
    if (nk > 0) {
        if constexpr (AMODE == 3) la.issue(A, 0, lds);
        if constexpr (BMODE == 3) lb.issue(B, 0, lds + A_BYTES);
        la.load(A, g.sak, 0, g.k);
        lb.load(B, g.sbk, 0, g.k);
        la.store(lds);
        lb.store(lds + A_BYTES);
    }
    __syncthreads();

    // Fragment reads are software-pipelined one K sub-step (16) ahead of the MFMAs that consume
    // them, and the barrier that publishes the next tile sits before the last sub-step, so the LDS
    // latency of the first fragments of tile t+1 hides behind the last MFMAs of tile t.
    const int frow = lane & 31, fk = lane >> 5;
    const int a_row = wm * WM + frow, b_row = wn * WN + frow;
    half8 af[2][TM], bf[2][TN];
    auto read_frags = [&](const char* buf, int kk, half8(&fa)[TM], half8(&fb)[TN]) {
        const int c = kk * 2 + fk;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int r = a_row + i * 32;
            fa[i] = *reinterpret_cast<const half8*>(buf + r * kRowBytes + ((c ^ swz(r)) << 4));
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int r = b_row + j * 32;
            fb[j] = *reinterpret_cast<const half8*>(buf + A_BYTES + r * kRowBytes + ((c ^ swz(r)) << 4));
        }
    };
    if (nk > 0) read_frags(lds, 0, af[0], bf[0]);
    for (int kt = 0; kt < nk; ++kt) {
        char* cur = lds + (kt & 1) * (A_BYTES + B_BYTES);
        char* nxt = lds + ((kt + 1) & 1) * (A_BYTES + B_BYTES);
        const bool more = kt + 1 < nk;
        if (more) {
            if constexpr (AMODE == 3) la.issue(A, (kt + 1) * BK, nxt);
            if constexpr (BMODE == 3) lb.issue(B, (kt + 1) * BK, nxt + A_BYTES);
            la.load(A, g.sak, (kt + 1) * BK, g.k);
            lb.load(B, g.sbk, (kt + 1) * BK, g.k);
        }
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            if (kk + 1 < BK / 16) {
                read_frags(cur, kk + 1, af[(kk + 1) & 1], bf[(kk + 1) & 1]);
            } else {
                if (more) {
                    la.store(nxt);
                    lb.store(nxt + A_BYTES);
                }
                __syncthreads();
                if (more) read_frags(nxt, 0, af[0], bf[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[kk & 1][j], af[kk & 1][i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();

    // ---- epilogue. With the swapped MFMA operands acc[i][j][e] is C[m, n] with m = l%32 and
    // n = (e/4)*8 + (l/32)*4 + e%4 inside the 32x32 block. Each wavefront stages one 32 x WN strip at a
    // time in its own LDS region and reads it back row-wise, so that global accesses are 128-bit and
    // contiguous along n.
    constexpr int PITCH = WN + 4;
    float* strip = reinterpret_cast<float*>(lds) + wave * 32 * PITCH;
    float bias_n[8];
    load_bias_n<WN>(g, bias_ptr, n0 + wn * WN, lane, bias_n);
    static_for<0, TM>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        stage_strip<TN, PITCH>(strip, acc[i], lane);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int mb = m0 + wm * WM + i * 32, nb = n0 + wn * WN;
        if (g.out_f32) store_strip<float, WN, ACT ? EPI_GENERAL_ACT : EPI_GENERAL>(g, c_ptr, pre_ptr, res_ptr, bias_ptr, bias_n, strip, mb, nb, coff, lane);
        else store_strip<_Float16, WN, ACT ? EPI_GENERAL_ACT : EPI_GENERAL>(g, c_ptr, pre_ptr, res_ptr, bias_ptr, bias_n, strip, mb, nb, coff, lane);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    });
}

// ---------------------------------------------------------------- host side
enum { CFG_128x128 = 0, CFG_256x128 = 1, CFG_256x256 = 2 };

template <int BM, int BN, int WM, int WN>
int launch_cfg(GemmArgs& g, const _Float16* pa, const _Float16* pb, void* pc, const void* pbias, const void* pres,
               void* ppre, int amode, int bmode, long long batch, hipStream_t st) {
    g.tiles_m = (g.m + BM - 1) / BM;
    g.tiles_n = (g.n + BN - 1) / BN;
    const long long total = (long long)g.tiles_m * g.tiles_n * batch;
    DML_REQUIRE(total <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f16: %lld workgroups exceed the grid limit", total);
    g.total_blocks = total;
    const size_t lds = (size_t)2 * (BM + BN) * kRowBytes;
#define DML_GEMM_CASE(AM, BMD)                                                                                \
    if (amode == AM && bmode == BMD) {                                                                        \
        auto kern = g.act != DMLHIP_ACT_NONE ? gemm_f16_kernel<BM, BN, WM, WN, AM, BMD, true>                  \
                                             : gemm_f16_kernel<BM, BN, WM, WN, AM, BMD, false>;                \
        if (lds > 64 * 1024) {                                                                                \
            hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                               (int)lds);                                                     \
            if (e != hipSuccess) {                                                                            \
                set_error("gemm_f16: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));        \
                return (int)e;                                                                                \
            }                                                                                                 \
        }                                                                                                     \
        hipLaunchKernelGGL(kern, (unsigned)total, kThreads, lds, st, pa, pb, pc, pbias, pres, ppre, g);                                      \
        return launch_status("gemm_f16");                                                                     \
    }
    DML_GEMM_CASE(0, 0)
    DML_GEMM_CASE(0, 1)
    DML_GEMM_CASE(1, 0)
    DML_GEMM_CASE(1, 1)
    if constexpr (BM == 128 && BN == 128) {
        DML_GEMM_CASE(2, 2)
    }
#undef DML_GEMM_CASE
    set_error("gemm_f16: no kernel for operand modes %d/%d", amode, bmode);
    return DMLHIP_ERR_UNSUPPORTED;
}

// 0 = K-contiguous, 1 = row-contiguous (both with 16-byte-aligned vectors, extents that are
// multiples of the vector length and 32-bit element offsets), 2 = anything else.
int operand_mode(const void* p, int64_t rows, int64_t k, int64_t s_row, int64_t s_k, const int64_t* sb,
                 const int64_t* batch) {
    bool bs_ok = true;
    for (int i = 0; i < 3; ++i)
        if (batch[i] > 1 && sb[i] % 8 != 0) bs_ok = false;
    if (!aligned16(p) || !bs_ok) return 2;
    if ((double)(rows - 1) * s_row + (double)(k + 64) * s_k > 2.0e9) return 2;
    if (s_k == 1 && s_row % 8 == 0 && k % 8 == 0) return 0;
    if (s_row == 1 && s_k % 8 == 0 && rows % 8 == 0) return 1;
    return 2;
}

// Estimated time in us of the configuration (*cfg) that is the fastest for a product of few tiles: fixed + (rounds of
// resident workgroups - 1) * round + tiles per compute unit * K steps * step, fitted to 330 products of encoder layers
// (24 - 2048 tokens, 512 - 1024 wide, every operand layout); its choice is within 1 % of the fastest configuration in the
// mean, 19 % at worst. Decided by it (us, 128-wide tiles / 64 x 64 / 32 x 32): 128 x 1024 x 4096 19 / 15 / 9; 651 x 1024 x 4096
// 24 / 17 / 23; 651 x 4096 x 1024 11 / 19 / 24; the K-concatenated 651 x 1024 x 3 * 1024 26 / 14 / 22.
// narrow: the 128 x 64 tile exists; pipe: the pipelined kernels do; general: so does the kernel that stages its operands in
// registers (*cfg = -1), which is what a ragged K otherwise has. Its line is from 190 products of K = 8 - 1000, us there and
// in the better of the two split ones: 1048 x 2432 x 48 6.5 / 12.3, 4960 x 1048 x 504 22 / 39, 3720 x 1536 x 1000 30 / 54,
// 480 x 4096 x 520 15 / 11, 608 x 4096 x 1000 26 / 22, 72 x 256 x 520 13 / 5.
double estimate_small(int64_t m, int64_t n, int64_t k, long long batch, int pairs, bool out_f32, bool narrow, bool pipe,
                      bool general, int* cfg) {
    struct Est { int cfg, bm, bn, resident; double fixed, round, step; };
    constexpr Est kEst[] = {{5, 128, 128, 1, 5.59, 5.36, 0.353}, {7, 128, 128, 2, 5.26, 5.36, 0.484},
                            {9, 128, 64, 2, 3.22, 1.86, 0.326},  {10, 64, 64, 1, 4.51, 3.35, 0.182},
                            {12, 32, 32, 2, 3.26, 1.81, 0.100},  {-1, 128, 128, 2, 5.6, 0.0, 0.9}};
    const double steps = (double)ceil_div(k, (int64_t)BK) * pairs;
    double best_us = 1e30;
    for (const Est& e : kEst) {
        if (e.cfg < 0 ? !general : (e.cfg == 9 && !narrow) || (e.cfg < 10 && !pipe)) continue;
        // an fp32 result is the same bits whatever the tile: one accumulation chain in K order, which a split K is not
        if (e.cfg >= 10 && out_f32 && pipe) continue;
        const double t = (double)ceil_div(ceil_div(m, (int64_t)e.bm) * ceil_div(n, (int64_t)e.bn) * batch, (int64_t)kCus);
        const double us = e.fixed + (ceil(t / e.resident) - 1) * e.round + t * steps * e.step;
        if (us < best_us) {
            *cfg = e.cfg;
            best_us = us;
        }
    }
    return best_us;
}

// Whether the workgroups that stay for several 256 x 256 tiles (gemm_f16_wide.h) beat the 128 x 128 tile, as times in us of
// fixed + tiles per compute unit * (steps * step + what writing a tile takes). A residual is read while nothing is multiplied,
// and the more compute units work the lower their clock. a_kc: A is K-contiguous, the 128 x 128 tile that of gemm_f16_wide.h.
// Over 110 products (700 - 16384 tokens, 512 - 4096 wide, B in either layout, groups, operand pairs, residuals) the faster of
// the two was missed once, by 1 %. Decided by it (us, 128 x 128 tiles / 256 x 256): 5041 x 2048 x 1024 30.3 / 28.4, three of
// 4144 x 1024 x 1024 37.1 / 28.0, three of 5532 x 1024 x 4096 147 / 161, 4860 x 1024 x 4096 56.7 / 73, 8230 x 1024 x 3072 67 / 60.
// Short loops have to be ahead by more: those with a residual, which two workgroups per compute unit read under each other's loops
// (16791 x 2048 x 768 80.5 / 86.7, 10647 x 2048 x 768 52.1 / 54.9, fp32 2967 x 3072 x 512 29.2 / 31.2), and eight steps with a third
// round that is nearly empty (16512 x 2048 x 512 52.2 / 56.5). Of 1740 products that it takes from two workgroups per compute unit, 0.83
// of the time there in the mean, none is more than 4 % slower.
bool wide_is_faster(long long t256, long long t128, int64_t k, int pairs, bool residual, bool a_kc, bool out_f32) {
    const double steps = (double)(k / BK) * pairs;
    const double t = (double)ceil_div(t256, (long long)kCus), s = (double)ceil_div(t128, (long long)kCus);
    const double full = (double)t256 / (t * kCus);
    const double ahead = t >= 3 && k <= 512 && !residual ? 0.9 : residual && k <= 1024 && t128 >= 2 * kCus ? (out_f32 ? 0.95 : 0.975) : 1.0;
    return 9.0 + t * steps * (1.0 + 0.35 * full * full) + (t - 1) * 6.0 + (residual ? t * 6.0 : 0.0) <
           ahead * (4.0 + s * ((a_kc ? 0.43 : 0.55) * steps + (residual ? 3.5 : 2.0)));
}

// Diagnostic switches (declared in the public header). Per calling thread, so that one thread pinning a configuration
// does not change what other threads launch.
thread_local int g_force_cfg = -1;  // pin the tile configuration
thread_local int g_last_cfg = -1;   // configuration of the last product, -1 = operands staged in registers
thread_local int g_direct_lds = 1;  // 0 forces the register-staged loaders
thread_local unsigned long long* g_trace = nullptr;  // per-workgroup clock readings of the pipelined kernel

}  // namespace
}  // namespace dml

using namespace dml;

extern "C" {

void dmlhip_debug_force_gemm_config(int cfg) { g_force_cfg = cfg; }
void dmlhip_debug_gemm_direct_lds(int on) { g_direct_lds = on; }
void dmlhip_debug_gemm_trace(void* buffer) { g_trace = (unsigned long long*)buffer; }
int dmlhip_debug_last_gemm_config() { return g_last_cfg; }
static std::atomic<long long> g_grouped_single_launches{0};
// Number of grouped calls that went out as ONE launch (tests check that grouping really happens).
long long dmlhip_debug_grouped_single_launches() { return g_grouped_single_launches.load(); }

struct GemmGroup {
    int count;
    const void* const* a;
    const void* const* b;
    void* const* c;            // unused with ksum
    const void* const* bias;   // unused with ksum
    bool ksum;                 // concatenate the groups along K into one output instead of running them side by side
};

// What is refused of a product whichever kernel would run it; the number of its batch entries in `batch`.
static int check_gemm_f16(const dmlhip_gemm_desc* d, long long& batch) {
    DML_REQUIRE(d, DMLHIP_ERR_NULL, "gemm_f16: NULL descriptor");
    DML_REQUIRE(d->m >= 0 && d->n >= 0 && d->k >= 0, DMLHIP_ERR_SHAPE, "gemm_f16: negative extent");
    DML_REQUIRE(d->m <= 2147483647 / 2 && d->n <= 2147483647 / 2 && d->k <= 2147483647 / 2, DMLHIP_ERR_SHAPE,
                "gemm_f16: extent exceeds 2^30");
    batch = 1;
    for (int i = 0; i < 3; ++i) {
        DML_REQUIRE(d->batch[i] >= 0 && d->batch[i] <= 2147483647, DMLHIP_ERR_SHAPE, "gemm_f16: bad batch extent");
        batch *= d->batch[i];
        DML_REQUIRE(batch <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f16: batch too large");
    }
    DML_REQUIRE(d->out_dtype == DMLHIP_F16 || d->out_dtype == DMLHIP_F32, DMLHIP_ERR_ENUM, "gemm_f16: bad out_dtype");
    DML_REQUIRE(d->bias_dtype == DMLHIP_F16 || d->bias_dtype == DMLHIP_F32, DMLHIP_ERR_ENUM,
                "gemm_f16: bad bias_dtype");
    DML_REQUIRE(valid_act(d->act), DMLHIP_ERR_ENUM, "gemm_f16: bad act");
    DML_REQUIRE(d->a_stride_m >= 0 && d->a_stride_k >= 0 && d->b_stride_k >= 0 && d->b_stride_n >= 0 &&
                    d->c_stride_m >= 0,
                DMLHIP_ERR_SHAPE, "gemm_f16: negative stride");
    DML_REQUIRE(d->c_stride_m >= d->n || d->m <= 1, DMLHIP_ERR_SHAPE, "gemm_f16: rows of C overlap (stride %lld < n)",
                (long long)d->c_stride_m);
    return 0;
}

// grp != nullptr: a / b / c / bias are those of group 0 (used for the layout checks, which the caller has made sure
// hold for every group); returns DMLHIP_ERR_UNSUPPORTED when the grouped launch is not possible.
static int run_gemm_f16(const dmlhip_gemm_desc* d, const void* a, const void* b, void* c, const void* bias,
                        const void* residual, void* pre_out, void* stream, const GemmGroup* grp = nullptr,
                        void* const* asum = nullptr, int asum_f32 = 0) {
    long long batch;
    if (int e = check_gemm_f16(d, batch)) return e;
    if (d->m == 0 || d->n == 0 || batch == 0) return 0;
    DML_REQUIRE(c, DMLHIP_ERR_NULL, "gemm_f16: NULL output");
    DML_REQUIRE(d->k == 0 || (a && b), DMLHIP_ERR_NULL, "gemm_f16: NULL operand");

    GemmArgs g;
    g.groups = 0;
    g.ksum = 0;
    g.trace = g_trace;
    g.asum = !grp && asum ? asum[0] : nullptr;
    g.asum_f32 = asum_f32;
    for (int i = 0; i < DMLHIP_GROUP_MAX; ++i) g.gasum[i] = grp && asum && i < grp->count ? asum[i] : nullptr;
    if (grp) {
        g.groups = grp->count;
        g.ksum = grp->ksum;
        if (!grp->ksum) batch *= grp->count;
        for (int i = 0; i < DMLHIP_GROUP_MAX; ++i) {
            const bool on = i < grp->count;
            g.ga[i] = on ? (const _Float16*)grp->a[i] : nullptr;
            g.gb[i] = on ? (const _Float16*)grp->b[i] : nullptr;
            g.gc[i] = on && !grp->ksum ? grp->c[i] : nullptr;
            g.gbias[i] = on && !grp->ksum && grp->bias ? grp->bias[i] : nullptr;
        }
    }
    g.m = (int)d->m; g.n = (int)d->n; g.k = (int)d->k;
    g.sam = d->a_stride_m; g.sak = d->a_stride_k; g.sbn = d->b_stride_n; g.sbk = d->b_stride_k;
    g.scm = d->c_stride_m;
    g.batch1 = (int)d->batch[1]; g.batch2 = (int)d->batch[2];
    for (int i = 0; i < 3; ++i) {
        g.sab[i] = d->a_stride_batch[i]; g.sbb[i] = d->b_stride_batch[i]; g.scb[i] = d->c_stride_batch[i];
    }
    g.alpha = d->alpha; g.beta = d->beta;
    g.out_f32 = d->out_dtype == DMLHIP_F32; g.bias_f32 = d->bias_dtype == DMLHIP_F32; g.act = d->act;
    g.bias_m = d->bias_along_m != 0;
    {
        // 128-bit accesses to C / pre_out / residual need 8-element granularity everywhere
        const int gran = 8;
        bool ok = aligned16(c) && (!residual || aligned16(residual)) && (!pre_out || aligned16(pre_out)) &&
                  d->c_stride_m % gran == 0;
        if (g.out_f32)
            ok = ok && (reinterpret_cast<uintptr_t>(c) % 32 == 0) &&
                 (!residual || reinterpret_cast<uintptr_t>(residual) % 32 == 0) &&
                 (!pre_out || reinterpret_cast<uintptr_t>(pre_out) % 32 == 0);
        for (int i = 0; i < 3; ++i)
            if (d->batch[i] > 1 && d->c_stride_batch[i] % gran != 0) ok = false;
        g.c_vec = ok;
    }

    int amode = d->k == 0 ? 0 : operand_mode(a, d->m, d->k, d->a_stride_m, d->a_stride_k, d->a_stride_batch, d->batch);
    int bmode = d->k == 0 ? 0 : operand_mode(b, d->n, d->k, d->b_stride_n, d->b_stride_k, d->b_stride_batch, d->batch);
    if (amode == 2 || bmode == 2) amode = bmode = 2;
    hipStream_t st = (hipStream_t)stream;

    int cfg = g_force_cfg;
    // Both operands vector-loadable and K a whole number of steps, or a weight gradient over any number of tokens: the fully
    // pipelined kernel. The kernel with K split over the wavefronts takes any K.
    const int ek = epilogue_kind(g, bias, residual, pre_out);
    const bool ragged = d->k % BK != 0;
    const bool vec = amode != 2 && d->k > 0 && g_direct_lds && ek != EPI_GENERAL_ACT;
    const bool pipe = vec && (!ragged || (amode == 1 && bmode == 1 && ek == EPI_PLAIN && !g.ksum));
    if (vec) {
        auto blocks = [&](int bm, int bn) { return (long long)ceil_div(d->m, bm) * ceil_div(d->n, bn) * batch; };
        const bool sums = g.asum || (grp && g.gasum[0]);
        // what the kernels of gemm_f16_wide.h take
        const bool wide = pipe && !ragged && !sums && g.beta == 0.f && g.act == DMLHIP_ACT_NONE && !pre_out && g.c_vec && d->n % 8 == 0 &&
                          (!bias || g.bias_m || aligned16(bias));
        const long long steps = (long long)(d->k / BK) * (g.ksum ? g.groups : 1);
        const bool extra = grp || asum;   // operand pairs / row sums: the 128 x 128 tile only
        const long long t256 = blocks(256, 256), t128 = blocks(128, 128);
        const long long slots256 = ceil_div(t256, (long long)kCus) * kCus, slots128 = ceil_div(t128, (long long)kCus) * kCus;
        bool narrow = false;   // the estimate found the 128 x 64 tile to be the fastest
        const bool full256 = !extra && t256 * 10 >= slots256 * 9;
        if (cfg < 0 && d->k >= 512 && wide && (full256 || wide_is_faster(t256, t128, d->k, g.ksum ? g.groups : 1, residual, amode == 0, g.out_f32))) {
            cfg = 13;
        } else if (cfg < 0 && d->k >= 512 && full256) {
            // What the kernel above does not take (activations, beta, rows that are not stored in vectors, a ragged K). The
            // 256 x 256 tile halves the bytes each compute unit pulls through L2 and LDS per MFMA (4096 x 4096 x 1024: 39 us
            // against 45 - 54 us for every 128-wide tile), as long as its tiles fill (nearly) every round of compute units.
            cfg = 4;
        } else if (cfg < 0 && t128 < 2 * kCus && t128 * 10 < slots128 * 9 && (!pipe || d->k >= 512 || t128 <= kCus)) {
            // rows of C that are not written in vectors hide what the general kernel's longer loop costs: one round only
            const bool general = !pipe && !extra && (g.c_vec || t128 > kCus);
            estimate_small(d->m, d->n, d->k, batch, g.ksum ? g.groups : 1, g.out_f32, !extra, pipe, general, &cfg);
            narrow = cfg == 9;
        }
        if (cfg < 0) {
            if (d->k < 512) {
                // a handful of K steps (the batched products of an unfused attention): bound by the epilogue, where two
                // resident workgroups per compute unit overlap one's stores with the other's loads. 361 tiles, K = 64 / 192, us on
                // 3, 7 and the 128 x 64 tile: 5.5 / 7.2, 5.8 / 7.1, 7.0 / 7.8
                cfg = t128 <= kCus ? 0 : d->k < 192 ? 3 : 7;
            } else if (d->k <= 1024 && t128 >= 2 * kCus) {
                // several rounds of short K loops (the grouped q / k / v projections: 768 tiles of 16 steps): with two
                // LDS stages instead of four, two workgroups share a compute unit and one's epilogue and first loads
                // overlap the other's loop. Tiles that stay (gemm_f16_wide.h) are faster beyond one round of such pairs where a
                // pair would be left half empty or the loop is not short; time of 14 over 7 with 8 / 12 / 16 steps: five rounds 0.98 / 0.93 /
                // 0.92 (just past the fourth, 8 steps, 1.01 - 1.04), nine with a residual 1.01 / 0.95 / 0.97; four rounds with 8 - 10 / 12 / 13 / 14 / 16
                // steps 1.05 - 1.02 / 0.98 / 0.97 / 0.97 / 0.92 - 0.98 (taken from sixteen on), of fp32 with a residual 1.05.
                const long long rounds = ceil_div(t128, (long long)kCus);
                const bool half = rounds % 2 && (steps >= 12 || (rounds <= 5 && (t128 - (rounds - 1) * kCus) * 6 >= kCus));
                const bool stay = wide && amode == 0 && t128 > 2 * kCus && (half || (steps >= 16 && !(residual && g.out_f32)));
                cfg = stay ? 14 : 7;
            } else if (!extra && d->k <= 1024 && t128 <= kCus && residual) {
                // a short K loop whose epilogue also reads a residual tile (4096 x 1024 x 1024: 20.3 - 21.1 against
                // 22.9 - 23.2 us): 128 x 64 tiles, two workgroups per compute unit, for the same overlap (without the
                // residual the two tiles are level: 18.2 us). Fewer than 231 tiles have been decided above, where the estimate knows
                // no residual: of 300 products with and without one none was slower than with this line for them
                cfg = 9;
            } else {
                // one 128 x 128 tile per compute unit, four LDS stages, interleaved loop: 5 - 20 % faster than the plain
                // loop on every product of the layer with 4096 x 1024 or 1024 x 4096 outputs
                cfg = 5;
            }
        }
        const _Float16 *pa = (const _Float16*)a, *pb = (const _Float16*)b;
        // The 128 x 128 tile of gemm_f16_wide.h in place of those of gemm_f16_pipe.h, from sixteen steps on; not for the products
        // that the estimate gives to 128 x 64 tiles, which are two per compute unit (960 x 2048 x 1024 9.4 us there, 11.0 here).
        // It starts with more steps on their way and reads a residual of fp16 ahead. Without one, up to a round of tiles needs
        // thirty-two steps, and seven eighths of a round unless they are those of several operand pairs. us on 5 / 14: 1371 x 2048 x 1024
        // 11.3 / 11.6, B row-contiguous 2844 x 768 x 3072 22.4 / 23.6, but 4764 x 768 x 3072 26.5 / 25.6; three of 317 x 2048 x 1024
        // 11.4 / 12.5; fp32 with residual 768 x 3072 x 1024 14.4 / 15.9; with a residual 1280 x 2048 x 1024 13.5 / 12.7, 2432 x 1024 x 4096
        // 30.4 / 29.3. (1300 products of up to a round that it takes: 0.935 of the time on 5 in the mean, three more
        // than 1.01.)
        // Nor for an A that the last-level cache does not hold: beyond 220 MB 0.98 in the mean, but three pairs of 11621 x 384 x 4096
        // 175 / 189, three of 9408 x 256 x 4096 79 / 86.
        const bool below = t128 <= kCus && !(residual && !g.out_f32) &&
                           (steps < 32 || (!g.ksum && t128 * 8 < kCus * 7));
        const bool beyond = 2e-6 * (double)d->m * (double)d->k * (grp ? grp->count : (int)batch) > 220.0;
        if (g_force_cfg < 0 && (cfg == 5 || (cfg == 9 && !narrow)) && wide && amode == 0 && steps >= 16 && t128 * 2 >= kCus && !below && !beyond)
            cfg = 14;
        g_last_cfg = cfg;
        if (cfg == 13 && wide && steps >= 3) return launch_wide256(g, pa, pb, c, bias, residual, amode, bmode, batch, st);
        if (cfg == 14 && wide && steps >= 5 && amode == 0) return launch_wide128(g, pa, pb, c, bias, residual, amode, bmode, batch, st);
        if (cfg == 13 || cfg == 14) g_last_cfg = cfg = cfg == 13 ? 4 : 5;
        if (cfg >= 10 && (!sums || amode == 1))
            return launch_split(g, pa, pb, c, bias, residual, pre_out, amode, bmode, cfg, batch, st);
        if (pipe && ragged) return launch_pipelined_ragged(g, pa, pb, c, bias, residual, pre_out, cfg, batch, st);
        if (pipe)
            return launch_pipelined(g, pa, pb, c, bias, residual, pre_out, amode == 1 ? 4 : 3, bmode == 1 ? 4 : 3, cfg, batch, st);
        if (g_force_cfg < 0) cfg = -1;
    }
    g_last_cfg = -1;
    if (grp || asum) return DMLHIP_ERR_UNSUPPORTED;  // only the pipelined kernel takes pointer groups / makes row sums
    if (cfg < 0 || cfg > 2) {
        // Largest tile that still yields at least one workgroup per CU.
        auto blocks = [&](int bm, int bn) { return (long long)ceil_div(d->m, bm) * ceil_div(d->n, bn) * batch; };
        if (blocks(256, 256) >= 256) cfg = CFG_256x256;
        else if (blocks(256, 128) >= 256) cfg = CFG_256x128;
        else cfg = CFG_128x128;
    }
    if (amode == 2) cfg = CFG_128x128;
    switch (cfg) {
        case CFG_256x256: return launch_cfg<256, 256, 128, 128>(g, (const _Float16*)a, (const _Float16*)b, c, bias, residual, pre_out, amode, bmode,
                                                   batch, st);
        case CFG_256x128: return launch_cfg<256, 128, 128, 64>(g, (const _Float16*)a, (const _Float16*)b, c, bias, residual, pre_out, amode, bmode,
                                                   batch, st);
        default: return launch_cfg<128, 128, 64, 64>(g, (const _Float16*)a, (const _Float16*)b, c, bias, residual, pre_out, amode, bmode,
                                                   batch, st);
    }
}

// Whether both operands of a product are read 16 bytes at a time (then the slices of a split K run on the pipelined kernel).
static bool vector_operands(const dmlhip_gemm_desc* d, const void* a, const void* b) {
    return g_direct_lds && operand_mode(a, d->m, d->k, d->a_stride_m, d->a_stride_k, d->a_stride_batch, d->batch) != 2 &&
           operand_mode(b, d->n, d->k, d->b_stride_n, d->b_stride_k, d->b_stride_batch, d->batch) != 2;
}

// Number of K slices of a plain product, in workgroups of their own with fp32 results that a second launch adds up (1 = none).
static int split_k_factor(const dmlhip_gemm_desc* d, bool vec) {
    if (!d || d->m <= 0 || d->n <= 0 || d->k < 1024 || d->batch[0] * d->batch[1] * d->batch[2] != 1) return 1;
    int s = 1;
    if (!vec) {
        // The kernel that stages its operands in registers has 128 x 128 tiles and a long step: slices until they fill the
        // chip (1024 x 30 x 1024, B of odd pitch: 144 us as one, 52 in four slices).
        const long long tiles = ceil_div(d->m, 128) * ceil_div(d->n, 128);
        while (tiles <= 128 && tiles * s * 2 <= kCus && d->k / (s * 2) >= 256 && d->k % (s * 2 * BK) == 0) s *= 2;
        return s;
    }
    // The smallest estimate of both launches, at most 16 MiB of slices. The sum takes 3 us, 0.3 per slice and its reads and the
    // slices' stores 2.4 TB/s, six times that for rows that are not stored in vectors. Unsplit, 64 x 64 and 32 x 32
    // tiles fall behind their estimate when K is long, more so where an XCD's tiles cover many rows of A (2048 x 512 x 4096
    // fp16 24 - 27 us, 512 x 2048 x 4096 16). Fitted to 840 products of 64 - 2048 rows and columns, K = 1024 - 65536,
    // both result types, 1 - 32 slices each. Decided by it (us, one / 2 / 4 / 8 / 16 slices): 512 x 512 x 16384 fp32 79 / 43 / 26 / 20 /
    // 22; 1024 x 1024 x 4096 fp32 24 / 20 / 22 / 27 / 37, fp16 18 in one launch; 256 x 256 x 4096 fp32 19 / 14 / 11 / 11 / 12.
    int cfg;
    const double steps = (double)d->k / 1024;
    double best = estimate_small(d->m, d->n, d->k, 1, 1, d->out_dtype == DMLHIP_F32, true, true, false, &cfg) *
                  (1.0 + (d->m >= 2 * d->n ? 0.2 : 0.1) * fmin(fmax(steps - 2.0, 0.0), 4.0));
    for (int t = 2; d->k % (t * BK) == 0 && d->k / t >= 256; t *= 2) {
        const double bytes = 4.0 * t * (double)d->m * (double)d->n;
        if (bytes > 16.0 * 1048576) break;
        const double us = estimate_small(d->m, d->n, d->k / t, t, 1, true, true, true, false, &cfg) + 3.0 + 0.3 * t +
                          bytes * (d->n % 8 ? 6.0 : 1.0) / 2.4e6;
        if (us >= 0.95 * best) continue;
        best = us;
        s = t;
    }
    return s;
}

static size_t split_k_bytes(const dmlhip_gemm_desc* d, int s) {
    return s > 1 ? (size_t)s * d->m * d->n * sizeof(float) : 0;
}

int dmlhip_debug_gemm_f16_slices(const dmlhip_gemm_desc* d) { return split_k_factor(d, d && vector_operands(d, nullptr, nullptr)); }

// for the call with whatever addresses the operands have
size_t dmlhip_gemm_f16_workspace_bytes(const dmlhip_gemm_desc* d) {
    const size_t any = split_k_bytes(d, split_k_factor(d, false));
    const size_t vec = d && vector_operands(d, nullptr, nullptr) ? split_k_bytes(d, split_k_factor(d, true)) : 0;
    return any > vec ? any : vec;
}

int dmlhip_gemm_f16_ws(const dmlhip_gemm_desc* d, const void* a, const void* b, void* c, const void* bias,
                       const void* residual, void* pre_out, void* workspace, size_t workspace_bytes, void* stream) {
    const bool plain = d && !bias && !residual && !pre_out && d->beta == 0.f && d->act == DMLHIP_ACT_NONE && a && b && c &&
                       workspace && d->c_stride_m == d->n;
    const int s = plain ? split_k_factor(d, vector_operands(d, a, b)) : 1;
    if (s <= 1 || workspace_bytes < split_k_bytes(d, s)) return run_gemm_f16(d, a, b, c, bias, residual, pre_out, stream);
    long long batch;
    if (int e = check_gemm_f16(d, batch)) return e;   // the slices' own result type is another
    // stage 1: batch slot 0 enumerates the K slices; partial C tiles are dense fp32 [s][m][n]
    dmlhip_gemm_desc p = *d;
    p.k = d->k / s;
    p.batch[0] = s;
    p.a_stride_batch[0] = p.k * d->a_stride_k;
    p.b_stride_batch[0] = p.k * d->b_stride_k;
    p.c_stride_batch[0] = d->m * d->n;
    p.c_stride_m = d->n;
    p.alpha = 1.f;
    p.out_dtype = DMLHIP_F32;
    if (int e = run_gemm_f16(&p, a, b, workspace, nullptr, nullptr, nullptr, stream)) return e;
    // stage 2: sum the slices, scale by alpha, convert
    const int64_t cols = d->m * d->n;
    hipStream_t st = (hipStream_t)stream;
    if (cols % 4 == 0) {
        int64_t blocks = ceil_div(cols / 4, 256);
        if (blocks > 256 * 16) blocks = 256 * 16;
        if (d->out_dtype == DMLHIP_F32)
            hipLaunchKernelGGL((sum_partials_vec4_kernel<float>), (unsigned)blocks, 256, 0, st, (const float*)workspace,
                               (float*)c, s, cols, cols, d->alpha);
        else
            hipLaunchKernelGGL((sum_partials_vec4_kernel<_Float16>), (unsigned)blocks, 256, 0, st,
                               (const float*)workspace, (_Float16*)c, s, cols, cols, d->alpha);
        return launch_status("gemm_f16(split-K sum)");
    }
    const unsigned grid = (unsigned)ceil_div(cols, kWave);
    if (d->out_dtype == DMLHIP_F32)
        hipLaunchKernelGGL((reduce_partials_kernel<OpSum, float>), grid, 1024, 0, st, (const float*)workspace, (float*)c,
                           s, cols, cols, 0.f, d->alpha, (float*)nullptr, (int64_t)0);
    else
        hipLaunchKernelGGL((reduce_partials_kernel<OpSum, _Float16>), grid, 1024, 0, st, (const float*)workspace,
                           (_Float16*)c, s, cols, cols, 0.f, d->alpha, (_Float16*)nullptr, (int64_t)0);
    return launch_status("gemm_f16(split-K sum)");
}

int dmlhip_gemm_f16(const dmlhip_gemm_desc* d, const void* a, const void* b, void* c, const void* bias,
                    const void* residual, void* pre_out, void* stream) {
    return run_gemm_f16(d, a, b, c, bias, residual, pre_out, stream);
}

int dmlhip_gemm_f16_grouped(const dmlhip_gemm_desc* d, int groups, const void* const* a, const void* const* b,
                            void* const* c, const void* const* bias, void* workspace, size_t workspace_bytes,
                            void* stream) {
    DML_REQUIRE(d, DMLHIP_ERR_NULL, "gemm_f16_grouped: NULL descriptor");
    DML_REQUIRE(groups >= 1 && groups <= DMLHIP_GROUP_MAX, DMLHIP_ERR_SHAPE, "gemm_f16_grouped: %d groups outside 1..%d",
                groups, DMLHIP_GROUP_MAX);
    DML_REQUIRE(a && b && c, DMLHIP_ERR_NULL, "gemm_f16_grouped: NULL pointer table");
    DML_REQUIRE(d->batch[0] == 1, DMLHIP_ERR_SHAPE, "gemm_f16_grouped: the outer batch extent must be 1");
    for (int i = 0; i < groups; ++i) DML_REQUIRE(c[i], DMLHIP_ERR_NULL, "gemm_f16_grouped: NULL output %d", i);
    // one launch when every group has the alignment of group 0 and the pipelined kernel applies
    bool same = d->k > 0 && d->beta == 0.f;
    for (int i = 0; i < groups && same; ++i) {
        same = a[i] && b[i] && aligned16(a[i]) && aligned16(b[i]) && reinterpret_cast<uintptr_t>(c[i]) % 32 == 0 &&
               (!bias == !(bias && bias[i])) && (!bias || aligned16(bias[i]));
    }
    if (same && groups > 1) {
        dmlhip_gemm_desc p = *d;
        p.a_stride_batch[0] = p.b_stride_batch[0] = p.c_stride_batch[0] = 0;   // the outer batch index selects the group
        GemmGroup grp = {groups, a, b, c, bias, false};
        const int e = run_gemm_f16(&p, a[0], b[0], c[0], bias ? bias[0] : nullptr, nullptr, nullptr, stream, &grp);
        if (e == 0) ++g_grouped_single_launches;
        if (e != DMLHIP_ERR_UNSUPPORTED) return e;
    }
    for (int i = 0; i < groups; ++i)
        if (int e = dmlhip_gemm_f16_ws(d, a[i], b[i], c[i], bias ? bias[i] : nullptr, nullptr, nullptr, workspace,
                                       workspace_bytes, stream))
            return e;
    return 0;
}

// Number of workgroups that share the K steps of a weight gradient's 256 x 256 tile (gemm_f16_wide.h); 0 = other kernels.
// How many: the fewest us of 9.5 + 1.4 per step + 0.3 per MB of partial results (written, read and summed). Whether at all: both
// launches take 20.6 us, 0.816 per step and 0.66 more where all compute units have a tile (0.038 more per 1024 columns beyond the
// first), 0.098 per MB (4.4 % off in the mean over 5656 gradients of 256 - 4096 x 256 - 4096 over 1000 - 18500 tokens, one to four
// products, both result types) - against 0.95 (a second round of less than 0.6: 0.86) of the 128 x 128 tiles' 4 + rounds * (2 + steps *
// (0.42 + 0.14 where all compute units have one)).
// us on those / here: 4096 x 1024 over 4096 / 8192 / 16384 tokens 42 / 51, 79 / 75, 153 / 122; 512 x 2048 over 4096 / 16384 34 / 31,
// 122 / 54; three of 1024 x 1024 over 16384 143 / 100; 896 x 896 over 3515 30.1 / 32.8, 256 x 640 over 1792 17.6 / 22.6.
// Results in fp16 may also be on the tiles with K split over the wavefronts, whose estimate long products exceed: 32 x 32 tiles by 1.3 - 2,
// 64 x 64 tiles by 1 - 1.2, and by 1.2 - 1.8 where the result has more rows than columns and a multiple of 512 of them.
// us there / here: 768 x 768 over 8128 tokens 31.4 / 34.2, over 10240 37.7 / 35.9; 384 x 1536 over 7872 26.6 / 36.1, 640 x 512 over 5540
// 22.4 / 29.0; 512 x 2048 over 4664 20.8 / 36.3, 2048 x 512 over 14283 84.9 / 49.6; 512 x 512 over 4160 15.4 / 28.8, over 14935 45.6 / 32.1.
// Of 12 440 gradients that may be faster here 12 255 go here; 52 of those are more than 2 % slower than there, 9 % at most.
static int weight_gradient_slices(const dmlhip_gemm_desc* d, int groups) {
    if (d->m <= 0 || d->n <= 0 || d->k <= 0 || d->m % 8 || d->n % 8 || d->c_stride_m != d->n || !g_direct_lds) return 0;
    if (d->m > 65536 || d->n > 65536 || (g_force_cfg >= 0 && g_force_cfg != 13)) return 0;
    const long long t256 = ceil_div(d->m, (int64_t)kWideTile) * ceil_div(d->n, (int64_t)kWideTile) * groups;
    const long long t128 = ceil_div(d->m, (int64_t)128) * ceil_div(d->n, (int64_t)128) * groups;
    // three steps each at least, four where the last one is ragged
    const long long steps = ceil_div(d->k, (int64_t)BK), least = d->k % BK ? 4 : 3;
    const long long most = steps / least < kCus / t256 ? steps / least : kCus / t256;
    if (most < 2) return 0;
    if (g_force_cfg == 13) return (int)most;
    const double mb = 4e-6 * groups * (double)d->m * (double)d->n;
    int slices = 0;
    double least_us = 1e30;
    for (int s = 2; s <= most; ++s) {
        const double us = 9.5 + 1.4 * (double)ceil_div(steps, (long long)s) + 0.3 * mb * s;
        if (us < least_us) {
            least_us = us;
            slices = s;
        }
    }
    const long long rounds = ceil_div(t128, (long long)kCus);
    const double tiles = 4.0 + (double)rounds * (2.0 + steps * (0.42 + 0.14 * fmin(1.0, t128 / (double)kCus)));
    double split = 1e30, behind = 1.0;
    if (d->out_dtype == DMLHIP_F16 && t128 < 2 * kCus && t128 * 10 < rounds * kCus * 9) {
        int cfg = -1;
        const double est = estimate_small(d->m, d->n, d->k, groups, 1, false, false, true, false, &cfg);
        const bool far = d->m % 512 == 0 && d->m > 512 && d->m > d->n;
        const bool many = ceil_div(d->m, (int64_t)64) * ceil_div(d->n, (int64_t)64) * groups >= 192;
        if (cfg >= 10) {
            split = est;
            behind = cfg == 12 ? 1.3 : far ? (many ? 1.3 : 1.18) : d->n >= 3 * d->m ? 0.92 : 1.02;
        }
    }
    const double full = (double)t256 * slices / kCus;
    const double wide_rows = d->n > 1024 ? 0.038 * (double)(d->n - 1024) / 1024 : 0.0;
    const double us = 20.6 + (double)ceil_div(steps, (long long)slices) * (0.816 + (0.66 + wide_rows) * full) + 0.098 * mb * slices;
    // the figures that the number of slices was chosen by have to say so too: those of many MB are the surer ones
    const bool faster = us < tiles * (rounds > 1 && t128 * 5 < rounds * kCus * 4 ? 0.86 : 0.95) && us < split * behind &&
                        least_us < tiles * 0.93 && least_us < split * 1.2;
    return faster ? slices : 0;
}

size_t dmlhip_gemm_f16_grouped_asum_workspace_bytes(const dmlhip_gemm_desc* d) {
    if (!d) return 0;
    const size_t g = dmlhip_gemm_f16_workspace_bytes(d);
    const size_t r = dmlhip_reduce_workspace_bytes(1, d->k, d->m);
    size_t most = g > r ? g : r, row_offset;
    for (int groups = 1; groups <= DMLHIP_GROUP_MAX; ++groups)
        if (const int s = weight_gradient_slices(d, groups)) {
            const size_t w = wide_sliced_bytes(d->m, d->n, groups, s, &row_offset);
            if (w > most) most = w;
        }
    return most;
}

int dmlhip_gemm_f16_grouped_asum(const dmlhip_gemm_desc* d, int groups, const void* const* a, const void* const* b,
                                 void* const* c, void* const* asum, int asum_dtype, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    DML_REQUIRE(d, DMLHIP_ERR_NULL, "gemm_f16_grouped_asum: NULL descriptor");
    DML_REQUIRE(groups >= 1 && groups <= DMLHIP_GROUP_MAX, DMLHIP_ERR_SHAPE,
                "gemm_f16_grouped_asum: %d groups outside 1..%d", groups, DMLHIP_GROUP_MAX);
    DML_REQUIRE(a && b && c && asum, DMLHIP_ERR_NULL, "gemm_f16_grouped_asum: NULL pointer table");
    DML_REQUIRE(asum_dtype == DMLHIP_F16 || asum_dtype == DMLHIP_F32, DMLHIP_ERR_ENUM,
                "gemm_f16_grouped_asum: bad asum_dtype");
    DML_REQUIRE(d->batch[0] == 1 && d->batch[1] == 1 && d->batch[2] == 1, DMLHIP_ERR_SHAPE,
                "gemm_f16_grouped_asum: batched products are not supported");
    DML_REQUIRE(d->beta == 0.f && d->act == DMLHIP_ACT_NONE, DMLHIP_ERR_UNSUPPORTED,
                "gemm_f16_grouped_asum: beta and activations are not supported");
    DML_REQUIRE(d->a_stride_m == 1 && d->a_stride_k == d->m, DMLHIP_ERR_UNSUPPORTED,
                "gemm_f16_grouped_asum: A must be stored as a dense [k, m] matrix");
    for (int i = 0; i < groups; ++i)
        DML_REQUIRE(c[i] && asum[i] && (d->k == 0 || (a[i] && b[i])), DMLHIP_ERR_NULL,
                    "gemm_f16_grouped_asum: NULL tensor in group %d", i);
    long long batch;
    if (int e = check_gemm_f16(d, batch)) return e;   // the products in slices below do not go through run_gemm_f16
    bool same = d->k > 0;
    for (int i = 0; i < groups && same; ++i)
        same = aligned16(a[i]) && aligned16(b[i]) && reinterpret_cast<uintptr_t>(c[i]) % 32 == 0;
    // A gradient over a ragged number of tokens that fills the chip with 256 x 256 tiles, which make no row sums: the product and
    // the sums one after the other. us here / in one launch on 128 x 128 tiles: 4096 x 4096 over 810 tokens 37 / 35, over 1233
    // 53 / 62, over 6689 192 / 260.
    if (groups == 1 && d->k % BK && d->k > 1024 && workspace_bytes >= dmlhip_reduce_workspace_bytes(1, d->k, d->m)) {
        const long long t256 = ceil_div(d->m, (int64_t)256) * ceil_div(d->n, (int64_t)256);
        if (t256 * 10 >= ceil_div(t256, (long long)kCus) * kCus * 9) same = false;
    }
    const int slices = same ? weight_gradient_slices(d, groups) : 0;
    if (slices) {
        const int64_t one[3] = {1, 1, 1};
        size_t row_offset;
        const int amode = operand_mode(a[0], d->m, d->k, d->a_stride_m, d->a_stride_k, d->a_stride_batch, one);
        const int bmode = operand_mode(b[0], d->n, d->k, d->b_stride_n, d->b_stride_k, d->b_stride_batch, one);
        if (amode == 1 && bmode != 2 && workspace && aligned16(workspace) &&
            workspace_bytes >= wide_sliced_bytes(d->m, d->n, groups, slices, &row_offset)) {
            GemmArgs g{};
            g.m = (int)d->m; g.n = (int)d->n; g.k = (int)d->k;
            g.sam = d->a_stride_m; g.sak = d->a_stride_k; g.sbn = d->b_stride_n; g.sbk = d->b_stride_k;
            g.alpha = d->alpha;
            g.out_f32 = d->out_dtype == DMLHIP_F32;
            g.c_vec = 1;
            g_last_cfg = 13;
            const _Float16 *ga[DMLHIP_GROUP_MAX], *gb[DMLHIP_GROUP_MAX];
            for (int i = 0; i < groups; ++i) {
                ga[i] = (const _Float16*)a[i];
                gb[i] = (const _Float16*)b[i];
            }
            return launch_wide_sliced(g, groups, slices, ga, gb, c, asum, asum_dtype == DMLHIP_F32, bmode, workspace,
                                      (hipStream_t)stream);
        }
    }
    if (same) {
        int e;
        if (groups > 1) {
            dmlhip_gemm_desc p = *d;
            p.a_stride_batch[0] = p.b_stride_batch[0] = p.c_stride_batch[0] = 0;
            GemmGroup grp = {groups, a, b, c, nullptr, false};
            e = run_gemm_f16(&p, a[0], b[0], c[0], nullptr, nullptr, nullptr, stream, &grp, asum, asum_dtype == DMLHIP_F32);
        } else {
            e = run_gemm_f16(d, a[0], b[0], c[0], nullptr, nullptr, nullptr, stream, nullptr, asum, asum_dtype == DMLHIP_F32);
        }
        if (e == 0) ++g_grouped_single_launches;
        if (e != DMLHIP_ERR_UNSUPPORTED) return e;
    }
    // products and column sums of the stored [k, m] matrices one after the other
    for (int i = 0; i < groups; ++i) {
        if (int e = dmlhip_gemm_f16_ws(d, a[i], b[i], c[i], nullptr, nullptr, nullptr, workspace, workspace_bytes, stream))
            return e;
        if (int e = dmlhip_reduce_f16(DMLHIP_RSUM, a[i], asum[i], asum_dtype, 1, d->k, d->m, workspace, workspace_bytes,
                                      stream))
            return e;
    }
    return 0;
}

int dmlhip_gemm_f16_ksum(const dmlhip_gemm_desc* d, int groups, const void* const* a, const void* const* b, void* c,
                         const void* bias, const void* residual, void* stream) {
    DML_REQUIRE(d, DMLHIP_ERR_NULL, "gemm_f16_ksum: NULL descriptor");
    DML_REQUIRE(groups >= 1 && groups <= DMLHIP_GROUP_MAX, DMLHIP_ERR_SHAPE, "gemm_f16_ksum: %d groups outside 1..%d",
                groups, DMLHIP_GROUP_MAX);
    DML_REQUIRE(a && b && c, DMLHIP_ERR_NULL, "gemm_f16_ksum: NULL pointer");
    DML_REQUIRE(d->beta == 0.f && d->act == DMLHIP_ACT_NONE, DMLHIP_ERR_UNSUPPORTED,
                "gemm_f16_ksum: beta and activations are not supported");
    for (int i = 0; i < groups; ++i) DML_REQUIRE(a[i] && b[i], DMLHIP_ERR_NULL, "gemm_f16_ksum: NULL operand %d", i);
    bool same = d->k > 0 && groups > 1;
    for (int i = 0; i < groups && same; ++i) same = aligned16(a[i]) && aligned16(b[i]);
    if (same) {
        GemmGroup grp = {groups, a, b, nullptr, nullptr, true};
        const int e = run_gemm_f16(d, a[0], b[0], c, bias, residual, nullptr, stream, &grp);
        if (e == 0) ++g_grouped_single_launches;
        if (e != DMLHIP_ERR_UNSUPPORTED) return e;
    }
    // one product after the other, accumulating in C (rounded to C's type in between)
    dmlhip_gemm_desc p = *d;
    for (int i = 0; i < groups; ++i) {
        if (int e = run_gemm_f16(&p, a[i], b[i], c, i == 0 ? bias : nullptr, i == 0 ? residual : nullptr, nullptr, stream))
            return e;
        p.beta = 1.f;
    }
    return 0;
}

}  // extern "C"
