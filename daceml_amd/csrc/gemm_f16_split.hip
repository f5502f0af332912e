// fp16 GEMM for products whose 128-wide tiles leave most of the 256 compute units idle (short sequences, single requests):
// tiles of 64 x 64 or 32 x 32 with K split over the four wavefronts of a workgroup.
//
// What bounds such a product is how fast a compute unit takes in its operands, not the matrix pipe: an M = 128 product over
// N = 1024, K = 4096 is 16 tiles of 128 x 64, and each of those 16 compute units pulls 1.5 MB through its own 64 bytes per
// clock while 240 others idle. Here every wavefront takes every fourth K step of the whole tile through a ring of its own
// in LDS (global_load_lds, no staging registers). Nothing is shared between the wavefronts inside the loop, so there is no
// barrier in it: a wavefront waits for its own transfers, reads the step's fragments, hands the stage back to the transfers
// and multiplies. The four partial tiles are added through LDS in a fixed order behind the loop.
// The last K step may be ragged: its missing part is transferred from a page of zeros.
#include "gemm_f16_common.h"

namespace dml {
namespace gemm16 {
namespace {

__device__ const half8 g_zeros = {0, 0, 0, 0, 0, 0, 0, 0};

// One operand of a wavefront: R = 32 T tile rows x 64 k per stage.
// KIND 0, K-contiguous: LDS rows of 64 k, 16-byte chunk c of row r at slot c ^ swz16(r), fragments by ds_read_b128.
// KIND 1, row-contiguous: LDS rows of one k, fragments by two transpose reads (see gemm_f16_pipe.h).
template <int T, int KIND> struct WaveStream;

template <int T>
struct WaveStream<T, 0> {
    static constexpr int R = 32 * T, N = R / 8;
    int off[N];
    int kl[2];                         // first k of this lane's chunk in even / odd transfers
    uint32_t faddr[4];
    __device__ __forceinline__ void init(int64_t s_row, int64_t, int row0, int rows, int lane, uint32_t tile0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int r = i * 8 + (lane >> 3);
            const int k = ((lane & 7) ^ swz16(r)) * 8;
            if (i < 2) kl[i] = k;
            off[i] = (int)(min(row0 + r, rows - 1) * s_row) + k;
        }
        const int r = lane & 31;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) faddr[kk] = tile0 + r * kRowBytes + (((kk * 2 + (lane >> 5)) ^ swz16(r)) << 4);
    }
    __device__ __forceinline__ int k_of(int i) const { return kl[i & 1]; }   // the swizzle repeats every 16 rows
    template <int KK>
    __device__ __forceinline__ void frags(uint32_t stage, half8 (&f)[T]) const {
        static_for<0, T>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            f[i] = lds_read_b128<i * 32 * kRowBytes>(faddr[KK] + stage);
        });
    }
};

template <int T>
struct WaveStream<T, 1> {
    static constexpr int R = 32 * T, N = R / 8, P = R * 2;
    int off[N];
    int kl0;
    uint32_t faddr[T];
    // K rows k and k + 2 of 128 bytes share their banks: shifted by half a row ((k / 2) % 2). 64-byte K rows do not collide.
    __device__ __forceinline__ static int shift(int k) { return T == 2 ? ((k >> 1) & 1) << 2 : 0; }
    __device__ __forceinline__ void init(int64_t, int64_t s_k, int row0, int rows, int lane, uint32_t tile0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int o = i * 1024 + lane * 16;
            const int k = o / P, c = ((o % P) >> 4) ^ shift(k);
            if (i == 0) kl0 = k;
            off[i] = (int)(k * s_k) + min(row0 + c * 8, rows - 8);
        }
        const int s = lane & 15, grp = lane >> 4;
        const int kq = (grp >> 1) * 8 + (s >> 2);
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const int row = i * 32 + (grp & 1) * 16 + 4 * (s & 3);
            faddr[i] = tile0 + kq * P + (((row >> 3) ^ shift(kq)) << 4) + (row & 7) * 2;
        }
    }
    __device__ __forceinline__ int k_of(int i) const { return kl0 + i * (1024 / P); }
    template <int KK>
    __device__ __forceinline__ void frags(uint32_t stage, half8 (&f)[T]) const {
        static_for<0, T>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const uint32_t a = faddr[i] + stage;
            const half4v lo = lds_read_tr16_b64<KK * 16 * P>(a);
            const half4v hi = lds_read_tr16_b64<KK * 16 * P + 4 * P>(a);
            f[i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        });
    }
};

template <typename S>
__device__ __forceinline__ void transfer(const S& s, const _Float16* p, int left, char* tile) {
    if (left >= BK) {
#pragma unroll
        for (int i = 0; i < S::N; ++i) lds_dma16(p + s.off[i], tile + i * 1024);
    } else {
#pragma unroll
        for (int i = 0; i < S::N; ++i)
            lds_dma16(s.k_of(i) < left ? p + s.off[i] : reinterpret_cast<const _Float16*>(&g_zeros), tile + i * 1024);
    }
}

// KSUM: operand pairs concatenated along K. ASUM: the workgroups of tile column 0 also add up the rows of A.
template <int T, int NSTAGE, int AKIND, int BKIND, int EPI, bool KSUM, bool ASUM>
__global__ __launch_bounds__(kThreads) void gemm_f16_split_kernel(const _Float16* a_ptr, const _Float16* b_ptr, void* c_ptr,
                                                                  const void* bias_ptr, const void* res_ptr, void* pre_ptr,
                                                                  const GemmArgs g) {
    constexpr int TB = 32 * T, TILE = TB * kRowBytes, STAGE = 2 * TILE, LPT = 2 * (TB / 8);
    extern __shared__ __attribute__((aligned(16))) char lds[];
    uint32_t bid = blockIdx.x;
    {
        const uint32_t total = (uint32_t)g.total_blocks;
        const uint32_t xcd = bid % kXcds, idx = bid / kXcds;
        const uint32_t base = total / kXcds, rem = total % kXcds;
        bid = xcd * base + (xcd < rem ? xcd : rem) + idx;
    }
    const uint32_t tiles = (uint32_t)(g.tiles_m * g.tiles_n);
    const uint32_t batch = bid / tiles, tile = bid - batch * tiles;
    // row tile fastest: the tiles an XCD works on together share columns of B, the weight, which is the larger operand here
    const int tn = (int)(tile / (uint32_t)g.tiles_m), tm = (int)(tile - (uint32_t)tn * (uint32_t)g.tiles_m);
    const uint32_t b2 = (uint32_t)g.batch2, b1 = (uint32_t)g.batch1, q = batch / b2;
    const int z2 = (int)(batch - q * b2), z0 = (int)(q / b1), z1 = (int)(q - (uint32_t)z0 * b1);
    void* asum_ptr = g.asum;
    if (!KSUM && g.groups) {
        a_ptr = g.ga[z0];
        b_ptr = g.gb[z0];
        c_ptr = g.gc[z0];
        bias_ptr = g.gbias[z0];
        asum_ptr = g.gasum[z0];
    }
    const int64_t aoff = z0 * g.sab[0] + z1 * g.sab[1] + z2 * g.sab[2];
    const int64_t boff = z0 * g.sbb[0] + z1 * g.sbb[1] + z2 * g.sbb[2];
    const int64_t coff = z0 * g.scb[0] + z1 * g.scb[1] + z2 * g.scb[2];
    const int m0 = tm * TB, n0 = tn * TB;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    char* const ring = lds + wave * NSTAGE * STAGE;
    const uint32_t ring0 = lds_addr(ring);

    floatx16 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    const bool do_asum = ASUM && tn == 0 && asum_ptr != nullptr;
    float acc_sum[ASUM ? T : 1];
    if constexpr (ASUM) {
#pragma unroll
        for (int i = 0; i < T; ++i) acc_sum[i] = 0.f;
    }

    WaveStream<T, AKIND> sa;
    WaveStream<T, BKIND> sb;
    sa.init(g.sam, g.sak, m0, g.m, lane, ring0);
    sb.init(g.sbn, g.sbk, n0, g.n, lane, ring0 + TILE);

    const int per_pair = (g.k + BK - 1) / BK;
    const int steps = KSUM ? per_pair * g.groups : per_pair;
    const int nk = (steps - wave + 3) / 4;             // steps wave, wave + 4, ...
    int fill_step = wave, pair = 0;                    // next step to transfer, inside its operand pair
    const _Float16* fa = a_ptr + aoff;
    const _Float16* fb = b_ptr + boff;
    auto fill = [&](int stage) {
        if constexpr (KSUM) {
            while (fill_step >= per_pair && pair + 1 < g.groups) {
                fill_step -= per_pair;
                ++pair;
                fa = (pair == 1 ? g.ga[1] : pair == 2 ? g.ga[2] : g.ga[3]) + aoff;
                fb = (pair == 1 ? g.gb[1] : pair == 2 ? g.gb[2] : g.gb[3]) + boff;
            }
        }
        const int k0 = fill_step * BK;
        transfer(sa, fa + (int64_t)k0 * g.sak, g.k - k0, ring + stage * STAGE);
        transfer(sb, fb + (int64_t)k0 * g.sbk, g.k - k0, ring + stage * STAGE + TILE);
        fill_step += 4;
    };
    static_assert(DMLHIP_GROUP_MAX == 4, "the operand-pair selection above lists four entries");
#pragma unroll
    for (int s = 0; s < NSTAGE; ++s)
        if (s < nk) fill(s);

    int stage = 0;
    for (int t = 0; t < nk; ++t) {
        // step t has landed; NSTAGE - 1 later ones stay in flight
        if (t + NSTAGE <= nk) wait_vm_lgkm0<(NSTAGE - 1) * LPT>();
        else wait_vm_lgkm0<0>();
        half8 af[4][T], bf[4][T];
        const uint32_t so = (uint32_t)stage * STAGE;
        static_for<0, 4>([&](auto kc) {
            constexpr int kk = decltype(kc)::value;
            sa.template frags<kk>(so, af[kk]);
            sb.template frags<kk>(so, bf[kk]);
        });
        wait_lgkm<0>();
        __builtin_amdgcn_sched_barrier(0);
        if (t + NSTAGE < nk) fill(stage);              // the fragments are in registers: the stage is free
        static_for<0, 4>([&](auto kc) {
            constexpr int kk = decltype(kc)::value;
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int j = 0; j < T; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[kk][j], af[kk][i], acc[i][j], 0, 0, 0);
            if constexpr (ASUM) {
                if (do_asum) {
                    const half2v one2 = {(_Float16)1.0f, (_Float16)1.0f};
#pragma unroll
                    for (int i = 0; i < T; ++i)
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            const half2v p = {af[kk][i][e], af[kk][i][e + 1]};
                            acc_sum[i] = __builtin_amdgcn_fdot2(p, one2, acc_sum[i], false);
                        }
                }
            }
        });
        stage = stage + 1 == NSTAGE ? 0 : stage + 1;
    }
    wait_vm_lgkm0<0>();
    __syncthreads();                                   // the rings are done with

    // Partial tiles as T x T blocks of 32 x 32 per wavefront, each a strip that store_strip can write out. With the MFMA
    // operands swapped a lane holds row lane % 32, columns 8 q + 4 (lane / 32) + 0 .. 3 of a block.
    constexpr int PITCH = 36, STRIP = 32 * PITCH;
    static_assert((4 * T * T * STRIP + 4 * TB) * 4 <= 4 * NSTAGE * STAGE, "the partial tiles fit the rings");
    float* const part = reinterpret_cast<float*>(lds);
    static_for<0, T>([&](auto ic) {
        static_for<0, T>([&](auto jc) {
            constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
            float* row = part + ((wave * T + i) * T + j) * STRIP + (lane & 31) * PITCH + (lane >> 5) * 4;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                *reinterpret_cast<floatx4*>(row + u * 8) =
                    floatx4{acc[i][j][4 * u], acc[i][j][4 * u + 1], acc[i][j][4 * u + 2], acc[i][j][4 * u + 3]};
        });
    });
    float* const hand = part + 4 * T * T * STRIP;      // [4 wavefronts][TB] row sums
    if constexpr (ASUM) {
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const int other = __builtin_amdgcn_ds_bpermute(((lane + 32) & 63) << 2, __builtin_bit_cast(int, acc_sum[i]));
            if (do_asum && lane < 32) hand[wave * TB + i * 32 + lane] = acc_sum[i] + __builtin_bit_cast(float, other);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < T * T; ++i) {
        float* p = part + i * STRIP + (threadIdx.x >> 3) * PITCH + (threadIdx.x & 7) * 4;
        floatx4 v = *reinterpret_cast<const floatx4*>(p);
#pragma unroll
        for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const floatx4*>(p + w * T * T * STRIP);
        *reinterpret_cast<floatx4*>(p) = v;
    }
    if constexpr (ASUM) {
        if (do_asum && threadIdx.x < TB && m0 + (int)threadIdx.x < g.m) {
            const float r = (hand[threadIdx.x] + hand[TB + threadIdx.x]) + (hand[2 * TB + threadIdx.x] + hand[3 * TB + threadIdx.x]);
            if (g.asum_f32) reinterpret_cast<float*>(asum_ptr)[m0 + threadIdx.x] = r;
            else reinterpret_cast<_Float16*>(asum_ptr)[m0 + threadIdx.x] = (_Float16)r;
        }
    }
    __syncthreads();
    if (wave < T * T) {
        const int mb = m0 + (wave / T) * 32, nb = n0 + (wave % T) * 32;
        float bias_n[8];
        load_bias_n<32>(g, bias_ptr, nb, lane, bias_n);
        const float* strip = part + wave * STRIP;
        if (g.out_f32) store_strip<float, 32, EPI>(g, c_ptr, pre_ptr, res_ptr, bias_ptr, bias_n, strip, mb, nb, coff, lane);
        else store_strip<_Float16, 32, EPI>(g, c_ptr, pre_ptr, res_ptr, bias_ptr, bias_n, strip, mb, nb, coff, lane);
    }
}

template <int T, int NSTAGE>
int launch_split_tile(GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* res, void* pre,
                      int ak, int bk, long long batch, hipStream_t st) {
    constexpr int TB = 32 * T;
    constexpr size_t lds = (size_t)4 * NSTAGE * 2 * TB * kRowBytes;
    g.tiles_m = (g.m + TB - 1) / TB;
    g.tiles_n = (g.n + TB - 1) / TB;
    const long long total = (long long)g.tiles_m * g.tiles_n * batch;
    DML_REQUIRE(total <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f16: %lld workgroups exceed the grid limit", total);
    g.total_blocks = total;
    const int ek = epilogue_kind(g, bias, res, pre);
    const bool sums = g.asum || (g.groups && g.gasum[0]);
#define DML_SPLIT(AK, BKD, EK, KS, AS)                                                                                   \
    if (ak == AK && bk == BKD && ek == EK && (bool)g.ksum == KS && sums == AS) {                                          \
        auto kern = gemm_f16_split_kernel<T, NSTAGE, AK, BKD, EK, KS, AS>;                                                \
        if (lds > 64 * 1024) {                                                                                            \
            const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
            if (e != hipSuccess) {                                                                                        \
                set_error("gemm_f16: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));                    \
                return (int)e;                                                                                            \
            }                                                                                                             \
        }                                                                                                                 \
        hipLaunchKernelGGL(kern, (unsigned)total, kThreads, lds, st, a, b, c, bias, res, pre, g);                         \
        return launch_status("gemm_f16(split)");                                                                          \
    }
#define DML_SPLIT_KINDS(EK, KS, AS) DML_SPLIT(0, 0, EK, KS, AS) DML_SPLIT(0, 1, EK, KS, AS) DML_SPLIT(1, 0, EK, KS, AS) DML_SPLIT(1, 1, EK, KS, AS)
    DML_SPLIT_KINDS(EPI_PLAIN, false, false)
    DML_SPLIT_KINDS(EPI_ACT, false, false)
    DML_SPLIT_KINDS(EPI_GENERAL, false, false)
    DML_SPLIT_KINDS(EPI_PLAIN, true, false)
    DML_SPLIT_KINDS(EPI_GENERAL, true, false)
    DML_SPLIT(1, 1, EPI_PLAIN, false, true)
    DML_SPLIT(1, 0, EPI_PLAIN, false, true)
#undef DML_SPLIT_KINDS
#undef DML_SPLIT
    set_error("gemm_f16: no split kernel for this product");
    return DMLHIP_ERR_UNSUPPORTED;
}

}  // namespace

int launch_split(GemmArgs& g, const _Float16* a, const _Float16* b, void* c, const void* bias, const void* residual, void* pre,
                 int ak, int bk, int cfg, long long batch, hipStream_t st) {
    if (cfg == 10) return launch_split_tile<2, 2>(g, a, b, c, bias, residual, pre, ak, bk, batch, st);
    return launch_split_tile<1, 2>(g, a, b, c, bias, residual, pre, ak, bk, batch, st);
}

}  // namespace gemm16
}  // namespace dml
