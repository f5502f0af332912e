// fp32 strided batched GEMM on v_mfma_f32_32x32x2_f32, operands streamed through LDS, for the fp32 MatMul / Einsum / Gemm nodes
// and the 1x1 convolutions: small and short products, and operands that cannot be read 16 bytes at a time (gemm_f32_split.hip has
// the entry point, the rule and the kernel for the others).
//
// What bounds it: the fp32 matrix rate (256 operations per clock and compute unit). A 64 x 64 tile needs 16 bytes per
// clock through L2 at that rate, a 32 x 32 tile 32 - both under the 64 that a compute unit takes in - so the tile is
// chosen for how evenly it spreads the problem over 256 compute units, not for operand reuse.
//
// Both operands go global -> LDS without staging registers (global_load_lds), K in steps of 32, into a ring of stages:
//   128 x 128   four wavefronts of 64 x 64 each, shared ring, one barrier per step; 4096^3 in 1032 us = 133 TFLOP/s
//   64 x 64     four wavefronts of 32 x 32 each, shared ring; three workgroups per compute unit
//   32 x 32     the four wavefronts take every fourth K step of the same tile, each with a ring of its own (no barrier in
//               the loop), and their sums are added through LDS behind it
// (A 128 x 128 tile staged through registers, whatever the problem, took 118 us for 1024 x 768 x 768 on its 48 workgroups;
// these take 20. Deeper rings, eight wavefronts with K split in two, and two accumulators per block measured no faster.)
// K-contiguous operands: LDS rows of 32 k (128 bytes, 16-byte chunks XOR-swizzled); a fragment read is one ds_read_b128
// whose four floats feed four successive MFMAs - which k of a step an MFMA multiplies is free as long as A and B agree.
// Row-contiguous operands: LDS rows of one k, fragments by ds_read_b32. Operands that cannot be read 16 bytes at a time
// (unaligned, odd pitch, any stride) are transferred 4 bytes per lane into the same two layouts. Lanes past the last row
// or the last k read a page of zeros instead, so every step issues the same transfers.
#include "common.h"
#include "lds_ops.h"

#include <type_traits>

namespace dml {
namespace {

constexpr int BK = 32;           // K per step
constexpr int kXcds = 8;
constexpr int kCus = 256;

// what lanes outside the operand read
__device__ const floatx4 g_zero_page = {0.f, 0.f, 0.f, 0.f};

struct GemmArgs32 {
    const float* a;
    const float* b;
    float* c;
    const void* bias;
    const float* residual;
    float* pre;
    int m, n, k;
    int64_t sam, sak, sbn, sbk, scm;
    int batch1, batch2;
    int64_t sab[3], sbb[3], scb[3];
    float alpha, beta;
    int bias_f32, act, bias_m;
    int tiles_m, tiles_n;
    int c_vec;                   // C (and residual, pre) can be accessed four columns at a time
    long long total_blocks;
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

// One operand: R tile rows x 32 k per stage, transferred by NW wavefronts, T blocks of 32 rows multiplied per wavefront.
// ROWS: 0 = LDS rows hold 32 k of one tile row, 1 = LDS rows hold R tile rows of one k. VEC: floats per lane and transfer.
template <int R, int NW, int T, int ROWS, int VEC>
struct Stream32 {
    static constexpr int PER = 64 * VEC;              // floats per transfer instruction
    static constexpr int N = R * BK / PER / NW;       // instructions per wavefront and step
    static_assert(N >= 1 && R * BK == N * NW * PER, "the tile is a whole number of transfers");
    // element offsets from the tile's first row, less than 2^29 for 16-byte pieces (the host checks): a transfer is then one
    // instruction with a scalar base. Lanes past the last row read the last one (they feed results that are not stored).
    typedef typename std::conditional<VEC == 4, uint32_t, int64_t>::type off_t;
    off_t off[N];
    int kl[N];          // k inside the step
    uint32_t faddr[ROWS ? 1 : 4];
    __device__ __forceinline__ void init(int64_t s_row, int64_t s_k, int rows_left, int wave, int lane, int wrow0, uint32_t tile0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int f = (i * NW + wave) * PER + lane * VEC;   // first float of this lane's piece in the LDS tile
            int r;
            if constexpr (ROWS == 0) {
                r = f / BK;
                kl[i] = ((((f % BK) >> 2) ^ (r & 7) ^ ((r >> 3) & 1)) << 2) + (f & 3);
                r = min(r, rows_left - 1);
            } else {
                r = min(f % R, rows_left - VEC);
                kl[i] = f / R;
            }
            off[i] = (off_t)((int64_t)r * s_row + (int64_t)kl[i] * s_k);
        }
        const int r = wrow0 + (lane & 31), half = lane >> 5;
        if constexpr (ROWS == 0) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk)
                faddr[kk] = tile0 + r * 128 + (((kk * 2 + half) ^ (r & 7) ^ ((r >> 3) & 1)) << 4);
        } else {
            faddr[0] = tile0 + (4 * half * R + r) * 4;
        }
    }
    // transfers [I0, I1) of a whole step from the step's first element
    template <int I0, int I1>
    __device__ __forceinline__ void issue(const float* p, char* tile, int wave) const {
        static_for<I0, I1>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            lds_dma<VEC * 4>(p + off[i], tile + (i * NW + wave) * PER * 4);
        });
    }
    // the same for a step that reaches past the end of K (`left` < 32, possibly none): zeros there
    template <int I0, int I1>
    __device__ __forceinline__ void issue_tail(const float* p, int left, char* tile, int wave) const {
        static_for<I0, I1>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            lds_dma<VEC * 4>(kl[i] < left ? p + off[i] : reinterpret_cast<const float*>(&g_zero_page),
                             tile + (i * NW + wave) * PER * 4);
        });
    }
    // fragments of k 8 KK .. 8 KK + 7: element j of block i is k = 8 KK + 4 (lane / 32) + j of row lane % 32
    template <int KK>
    __device__ __forceinline__ void frags(uint32_t stage, floatx4 (&f)[T]) const {
        static_for<0, T>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            if constexpr (ROWS == 0) {
                f[i] = __builtin_bit_cast(floatx4, lds_read_b128<i * 32 * 128>(faddr[KK] + stage));
            } else {
                const uint32_t a = faddr[0] + stage;
                f[i][0] = lds_read_b32<((KK * 8 + 0) * R + i * 32) * 4>(a);
                f[i][1] = lds_read_b32<((KK * 8 + 1) * R + i * 32) * 4>(a);
                f[i][2] = lds_read_b32<((KK * 8 + 2) * R + i * 32) * 4>(a);
                f[i][3] = lds_read_b32<((KK * 8 + 3) * R + i * 32) * 4>(a);
            }
        });
    }
};

// v = alpha * acc + bias, stored to pre; act(v) + residual + beta * C
__device__ __forceinline__ float finish(const GemmArgs32& g, float acc, float bias, int64_t off) {
    float v = g.alpha * acc + bias;
    if (g.pre) g.pre[off] = v;
    v = apply_act(g.act, v);
    if (g.residual) v += g.residual[off];
    if (g.beta != 0.f) v += g.beta * g.c[off];
    return v;
}

__device__ __forceinline__ float bias_at(const GemmArgs32& g, int i) {
    return g.bias_f32 ? reinterpret_cast<const float*>(g.bias)[i] : (float)reinterpret_cast<const _Float16*>(g.bias)[i];
}

// T: 32-row blocks per wavefront in each direction. WPG: wavefronts that share a tile and its ring (1 or 4). KG: groups of
// such wavefronts, each taking every KG-th K step of the tile.
template <int T, int WPG, int KG, int NSTAGE, int AROWS, int AVEC, int BROWS, int BVEC>
__global__ __launch_bounds__(kWave * WPG * KG) void gemm_f32_kernel(GemmArgs32 g) {
    static_assert(WPG == 1 || WPG == 4, "one wavefront or two by two");
    constexpr int TB = (WPG == 4 ? 64 : 32) * T;      // tile rows and columns
    constexpr int A_BYTES = TB * BK * 4, STAGE = 2 * A_BYTES;
    typedef Stream32<TB, WPG, T, AROWS, AVEC> SA;
    typedef Stream32<TB, WPG, T, BROWS, BVEC> SB;
    constexpr int LPT = SA::N + SB::N;                // transfers per wavefront and step
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
    // groups of eight tile rows, column by column: the tiles an XCD works on together share few rows and columns
    constexpr uint32_t kGroupM = 8;
    const uint32_t per_group = kGroupM * (uint32_t)g.tiles_n;
    const uint32_t group = tile / per_group, in_group = tile - group * per_group;
    const uint32_t rows_here = min((uint32_t)g.tiles_m - group * kGroupM, kGroupM);
    const int tn = (int)(in_group / rows_here), tm = (int)(group * kGroupM + in_group % rows_here);
    const int z2 = (int)(batch % (uint32_t)g.batch2);
    const uint32_t q = batch / (uint32_t)g.batch2;
    const int z1 = (int)(q % (uint32_t)g.batch1), z0 = (int)(q / (uint32_t)g.batch1);
    const float* A = g.a + z0 * g.sab[0] + z1 * g.sab[1] + z2 * g.sab[2];
    const float* B = g.b + z0 * g.sbb[0] + z1 * g.sbb[1] + z2 * g.sbb[2];
    const int64_t coff = z0 * g.scb[0] + z1 * g.scb[1] + z2 * g.scb[2];
    const int m0 = tm * TB, n0 = tn * TB;

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int kg = wave / WPG, sub = wave % WPG;      // K group, place in it
    const int wm = WPG == 4 ? (sub >> 1) * 32 * T : 0, wn = WPG == 4 ? (sub & 1) * 32 * T : 0;
    char* const ring = lds + kg * NSTAGE * STAGE;
    const uint32_t ring0 = lds_addr(ring);

    floatx16 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    A += m0 * g.sam;
    B += n0 * g.sbn;
    SA sa;
    SB sb;
    sa.init(g.sam, g.sak, g.m - m0, sub, lane, wm, ring0);
    sb.init(g.sbn, g.sbk, g.n - n0, sub, lane, wn, ring0 + A_BYTES);

    // Every group runs the same number of steps (the barriers are the workgroup's); a step past the end of K is all zeros.
    const int nk = ((g.k + BK - 1) / BK + KG - 1) / KG;
    auto issue = [&](int t, int stage, auto part_c, auto parts_c) {   // part of the transfers of step t
        constexpr int P = decltype(part_c)::value, OF = decltype(parts_c)::value;
        constexpr int A0 = P * SA::N / OF, A1 = (P + 1) * SA::N / OF, B0 = P * SB::N / OF, B1 = (P + 1) * SB::N / OF;
        const int k0 = (t * KG + kg) * BK;
        const float* pa = A + (int64_t)k0 * g.sak;
        const float* pb = B + (int64_t)k0 * g.sbk;
        char* at = ring + stage * STAGE;
        char* bt = at + A_BYTES;
        if (k0 + BK <= g.k) {
            sa.template issue<A0, A1>(pa, at, sub);
            sb.template issue<B0, B1>(pb, bt, sub);
        } else {
            sa.template issue_tail<A0, A1>(pa, g.k - k0, at, sub);
            sb.template issue_tail<B0, B1>(pb, g.k - k0, bt, sub);
        }
    };
    typedef std::integral_constant<int, 0> i0;
    typedef std::integral_constant<int, 1> i1;
    typedef std::integral_constant<int, 2> i2;
    floatx4 af[2][T], bf[2][T];
    int stage = 0;
    // One K step of four sub-steps. Reads of the next sub-step, the barrier and the refill of the ring all issue behind
    // MFMAs that are already queued. MORE: another step follows, whose first fragments are read under the last sub-step.
    auto step = [&](int t, auto more_c) {
        constexpr bool MORE = decltype(more_c)::value;
        const uint32_t so = (uint32_t)stage * STAGE;
        const int nxt = stage + 1 == NSTAGE ? 0 : stage + 1;
        static_for<0, 4>([&](auto kc) {
            constexpr int kk = decltype(kc)::value;
            constexpr int nb = (kk + 1) & 1;
            wait_lgkm<0>();
            __builtin_amdgcn_sched_barrier(0);
            static_for<0, 4>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
#pragma unroll
                for (int i = 0; i < T; ++i)
#pragma unroll
                    for (int j = 0; j < T; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[kk & 1][i][e], bf[kk & 1][j][e], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (kk < 3 && e == 0) {
                    sa.template frags<kk + 1>(so, af[nb]);
                    sb.template frags<kk + 1>(so, bf[nb]);
                } else if constexpr (kk == 3 && MORE && e == 0) {
                    // Every fragment of this step is in registers, so behind the barrier its stage is free and step t + 1
                    // has landed for all wavefronts of the ring.
                    if (t + NSTAGE - 1 < nk) wait_vm_lgkm0<(NSTAGE - 2) * LPT>();
                    else wait_vm_lgkm0<0>();
                    if constexpr (WPG > 1) __builtin_amdgcn_s_barrier();
                    sa.template frags<0>((uint32_t)nxt * STAGE, af[nb]);
                    sb.template frags<0>((uint32_t)nxt * STAGE, bf[nb]);
                } else if constexpr (kk == 3 && MORE && e == 1) {
                    if (t + NSTAGE < nk) issue(t + NSTAGE, stage, i0{}, i2{});
                } else if constexpr (kk == 3 && MORE && e == 2) {
                    if (t + NSTAGE < nk) issue(t + NSTAGE, stage, i1{}, i2{});
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        stage = nxt;
    };
    // one branch round all of it: a path on which the last step, which multiplies what was read ahead, is missing would leave
    // those reads unused (lds_ops.h)
    if (nk > 0) {
#pragma unroll
        for (int s = 0; s < NSTAGE; ++s)
            if (s < nk) issue(s, s, i0{}, i1{});
        if (NSTAGE <= nk) wait_vm_lgkm0<(NSTAGE - 1) * LPT>();
        else wait_vm_lgkm0<0>();
        if constexpr (WPG > 1) __builtin_amdgcn_s_barrier();
        sa.template frags<0>(0u, af[0]);
        sb.template frags<0>(0u, bf[0]);
        for (int t = 0; t + 1 < nk; ++t) step(t, std::true_type{});
        step(nk - 1, std::false_type{});
    }
    wait_vm_lgkm0<0>();

    // element e of a block: row (e / 4) * 8 + (lane / 32) * 4 + e % 4, column lane % 32
    if constexpr (KG > 1) {
        static_assert(T == 1, "one block per wavefront");
        constexpr int PITCH = TB + 4;                 // floats; rows stay 16-byte aligned and 4 banks apart
        static_assert(KG * TB * PITCH * 4 <= KG * NSTAGE * STAGE, "the partial tiles fit the rings");
        __syncthreads();                              // the rings are done with
        float* part = reinterpret_cast<float*>(lds);
#pragma unroll
        for (int e = 0; e < 16; ++e)
            part[(kg * TB + wm + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3)) * PITCH + wn + (lane & 31)] = acc[0][0][e];
        __syncthreads();
        constexpr int CPR = TB / 4;                   // pieces of four columns per row
        for (int i = threadIdx.x; i < TB * CPR; i += kWave * WPG * KG) {
            const int r = i / CPR, c4 = (i % CPR) * 4;
            const int m = m0 + r, n = n0 + c4;
            if (m >= g.m || n >= g.n) continue;
            floatx4 v = *reinterpret_cast<const floatx4*>(part + r * PITCH + c4);
#pragma unroll
            for (int w = 1; w < KG; ++w) v += *reinterpret_cast<const floatx4*>(part + (w * TB + r) * PITCH + c4);
            const int64_t off = coff + (int64_t)m * g.scm + n;
            const int cnt = min(4, g.n - n);
            const float bm = g.bias && g.bias_m ? bias_at(g, m) : 0.f;
            floatx4 out;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < cnt) out[e] = finish(g, v[e], g.bias && !g.bias_m ? bias_at(g, n + e) : bm, off + e);
            if (g.c_vec && cnt == 4) {
                *reinterpret_cast<floatx4*>(g.c + off) = out;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (e < cnt) g.c[off + e] = out[e];
            }
        }
    } else {
        const bool plain = !g.pre && g.act == DMLHIP_ACT_NONE && !g.residual && g.beta == 0.f && !(g.bias && g.bias_m);
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const int n = n0 + wn + j * 32 + (lane & 31);
            if (n >= g.n) continue;
            const float bias_n = g.bias && !g.bias_m ? bias_at(g, n) : 0.f;
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const int mb = m0 + wm + i * 32 + (lane >> 5) * 4;
                float* p = g.c + coff + (int64_t)mb * g.scm + n;
                if (plain) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int r = (e >> 2) * 8 + (e & 3);
                        if (mb + r < g.m) p[r * g.scm] = g.alpha * acc[i][j][e] + bias_n;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int r = (e >> 2) * 8 + (e & 3);
                        if (mb + r < g.m)
                            p[r * g.scm] = finish(g, acc[i][j][e], g.bias && g.bias_m ? bias_at(g, mb + r) : bias_n,
                                                  coff + (int64_t)(mb + r) * g.scm + n);
                    }
                }
            }
        }
    }
}

template <int T, int WPG, int KG, int NSTAGE, int AROWS, int AVEC, int BROWS, int BVEC>
int launch32(GemmArgs32& g, long long batch, hipStream_t st) {
    constexpr int TB = (WPG == 4 ? 64 : 32) * T;
    constexpr size_t lds = (size_t)NSTAGE * 2 * TB * BK * 4 * KG;
    g.tiles_m = (g.m + TB - 1) / TB;
    g.tiles_n = (g.n + TB - 1) / TB;
    const long long total = (long long)g.tiles_m * g.tiles_n * batch;
    DML_REQUIRE(total <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f32: too many workgroups");
    g.total_blocks = total;
    auto kern = gemm_f32_kernel<T, WPG, KG, NSTAGE, AROWS, AVEC, BROWS, BVEC>;
    if constexpr (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            set_error("gemm_f32: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
            return (int)e;
        }
    }
    hipLaunchKernelGGL(kern, (unsigned)total, kWave * WPG * KG, lds, st, g);
    return launch_status("gemm_f32");
}

template <int AROWS, int AVEC, int BROWS, int BVEC>
int launch_operands(GemmArgs32& g, int tile, long long batch, hipStream_t st) {
    if constexpr (AVEC == 4 && BVEC == 4) {
        if (tile == 0) return launch32<2, 4, 1, 2, AROWS, AVEC, BROWS, BVEC>(g, batch, st);
    }
    if (tile <= 1) return launch32<1, 4, 1, 3, AROWS, AVEC, BROWS, BVEC>(g, batch, st);
    return launch32<1, 1, 4, 2, AROWS, AVEC, BROWS, BVEC>(g, batch, st);
}

// How an operand is read: bit 0 = LDS rows of one k (row-contiguous in memory), bit 1 = 4 bytes per lane.
int operand_mode32(const void* p, int64_t rows, int64_t k, int64_t s_row, int64_t s_k, const int64_t* sb,
                   const int64_t* batch) {
    bool vec = aligned16(p) && 128.0 * s_row + 32.0 * s_k < 536870912.0;   // offsets inside a tile and step
    for (int i = 0; i < 3; ++i)
        if (batch[i] > 1 && sb[i] % 4 != 0) vec = false;
    if (s_k == 1) return vec && s_row % 4 == 0 && k % 4 == 0 ? 0 : 2;
    if (s_row == 1 && vec && s_k % 4 == 0 && rows % 4 == 0) return 1;
    return 3;
}

// The tile with the least estimated time. A compute unit works through its share of the tiles one K step after the other
// (workgroups that are resident together share its matrix pipes), and every round of resident workgroups adds its first
// loads and its stores. Measured step times: 1.93 / 0.56 / 0.155 us for 32 k of a 128 / 64 / 32 tile (31 / 34 / 39 ns per
// MFMA: the smaller the tile, the more instructions beside each MFMA). What it decides, us for the three tiles:
// 4096^3 1032 / 1124 / 1311; 1024 x 3072 x 768 (m x n x k) 62 / 51 / 63; 1024 x 768 x 3072 197 / 64 / 55;
// 64 x 128 x 784 58 / 19 / 8.
int choose_tile(int64_t m, int64_t n_cols, int64_t k, long long batch, double* estimate) {
    struct Tile { int size, resident; double round_us, step_us; };
    constexpr Tile kTiles[3] = {{128, 2, 8.0, 1.93}, {64, 3, 4.5, 0.56}, {32, 2, 4.5, 0.155}};
    const double steps = (double)ceil_div(k, (int64_t)BK);
    int best = 0;
    double best_t = 0;
    for (int i = 0; i < 3; ++i) {
        const Tile& t = kTiles[i];
        const double n = ceil((double)ceil_div(m, t.size) * ceil_div(n_cols, t.size) * batch / kCus);
        const double us = ceil(n / t.resident) * t.round_us + n * steps * t.step_us;
        if (i == 0 || us < best_t) {
            best = i;
            best_t = us;
        }
    }
    if (estimate) *estimate = best_t;
    return best;
}

}  // namespace

// What the chosen tile is estimated to take
double gemm_f32_streamed_us(const dmlhip_gemm_desc* d, long long batch) {
    double us;
    choose_tile(d->m, d->n, d->k, batch, &us);
    return us;
}

// The arguments are checked (gemm_f32_split.hip). tile: 0 = 128 x 128, 1 = 64 x 64, 2 = 32 x 32, -1: chosen here.
int gemm_f32_streamed(const dmlhip_gemm_desc* d, const void* a, const void* b, void* c, const void* bias, const void* residual,
                      void* pre_out, int tile, long long batch, hipStream_t st) {
    GemmArgs32 g;
    g.a = (const float*)a; g.b = (const float*)b; g.c = (float*)c;
    g.bias = bias; g.residual = (const float*)residual; g.pre = (float*)pre_out;
    g.m = (int)d->m; g.n = (int)d->n; g.k = (int)d->k;
    g.sam = d->a_stride_m; g.sak = d->a_stride_k; g.sbn = d->b_stride_n; g.sbk = d->b_stride_k; g.scm = d->c_stride_m;
    g.batch1 = (int)d->batch[1]; g.batch2 = (int)d->batch[2];
    for (int i = 0; i < 3; ++i) {
        g.sab[i] = d->a_stride_batch[i]; g.sbb[i] = d->b_stride_batch[i]; g.scb[i] = d->c_stride_batch[i];
    }
    g.alpha = d->alpha; g.beta = d->beta;
    g.bias_f32 = d->bias_dtype == DMLHIP_F32; g.act = d->act;
    g.bias_m = d->bias_along_m != 0;
    g.c_vec = aligned16(c) && d->c_stride_m % 4 == 0;
    for (int i = 0; i < 3; ++i)
        if (d->batch[i] > 1 && d->c_stride_batch[i] % 4 != 0) g.c_vec = 0;
    const int am = operand_mode32(a, d->m, d->k, d->a_stride_m, d->a_stride_k, d->a_stride_batch, d->batch);
    const int bm = operand_mode32(b, d->n, d->k, d->b_stride_n, d->b_stride_k, d->b_stride_batch, d->batch);
    if (tile < 0) tile = choose_tile(g.m, g.n, g.k, batch, nullptr);
#define DML_G32(AM, BMD) \
    if (am == AM && bm == BMD) \
        return launch_operands<(AM) & 1, (AM) & 2 ? 1 : 4, (BMD) & 1, (BMD) & 2 ? 1 : 4>(g, tile, batch, st);
    DML_G32(0, 0) DML_G32(0, 1) DML_G32(0, 2) DML_G32(0, 3)
    DML_G32(1, 0) DML_G32(1, 1) DML_G32(1, 2) DML_G32(1, 3)
    DML_G32(2, 0) DML_G32(2, 1) DML_G32(2, 2) DML_G32(2, 3)
    DML_G32(3, 0) DML_G32(3, 1) DML_G32(3, 2) DML_G32(3, 3)
#undef DML_G32
    return DMLHIP_ERR_UNSUPPORTED;
}

}  // namespace dml
