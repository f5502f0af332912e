// fp32 strided batched GEMM on the bf16 matrix cores: the entry point of the fp32 products and the kernel behind most of them.
//
// Operands are split into three bf16 values each (bf16_split.h has what that costs and keeps); K is cut into four or eight chains
// on top: 1024 x 768 x 768 is 0.8e-7 from the fp64 product where the streamed tiles are 2.5e-7 - 5.0e-7. Behind a ReLU and where nothing is
// negative errors are 0.08 - 0.67 of theirs, K of 256 - 65536. A wavefront whose sums come out not finite computes them again on the
// fp32 instruction.
//
// What bounds it: vector issue beside the matrix pipe. A wavefront's 64 x 64 tile is 24 MFMAs per 16 k (0.36 us) and 208
// instructions that split the operands; on a compute unit with eight wavefronts a step takes 0.57 us per wavefront and SIMD. So the
// splitting of the next step is placed between the MFMAs of this one (all of it first, then the MFMAs: 0.8 us). The sums of the large and
// the small products, two sets of pieces and the values read ahead are 240 of 256 registers: transfers share one or two offsets per
// operand, and the lane's number is found again where it is needed (four registers of offsets kept in scratch memory: 1024 x 768 x 3072 42.9 us
// instead of 39.7). Measured, us, the kernel of gemm_f32.hip / here: 1024 x 768 x 768 20 / 16, 1024 x 3072 x 768 51 / 39, 1024 x 768 x 3072 52 / 40,
// 3072 x 768 x 1024 (both operands row-contiguous) 59 / 43, 768 x 768 x 16384 (same) 244 / 148, 2048^3 136 / 115, 4096^3 1016 / 850. With all
// products in one sum, 1.0 - 1.6 times the error of the fp32 instruction where operands are half zero, these take 1 - 7 % less (15, 38, 38, 42, 146, 112).
#include "bf16_split.h"
#include "lds_ops.h"

#include <type_traits>

namespace dml {

int gemm_f32_streamed(const dmlhip_gemm_desc* d, const void* a, const void* b, void* c, const void* bias, const void* residual,
                      void* pre_out, int tile, long long batch, hipStream_t st);
double gemm_f32_streamed_us(const dmlhip_gemm_desc* d, long long batch);

namespace {

constexpr int BK = 16;           // K per step of a wavefront
constexpr int kXcds = 8;
constexpr int kBlock = 64;       // rows and columns of a tile
constexpr int kStages = 2;
constexpr int kCus = 256;

struct SplitArgs {
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

// The lane's number found again: a register less that the loop has to keep
__device__ __forceinline__ int lane_again() {
    uint32_t all = ~0u;
    asm volatile("" : "+s"(all));
    return (int)__builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0));
}

// what lanes outside the operand read
__device__ const floatx4 g_zero_page = {0.f, 0.f, 0.f, 0.f};

// One operand of a wavefront: 64 rows x 16 k per stage of its ring, 16 bytes per lane and transfer.
// ROWS = 0: LDS rows of 16 k (64 bytes, 16-byte chunks XOR-swizzled), block b of 32 has rows 32 b + j.
// ROWS = 1: LDS rows of one k, 64 tile rows each; block b has rows 2 j + b, so that one read fetches both blocks' values.
// Lanes past the last row read it again (their results are not stored), lanes past the last k a page of zeros.
template <int ROWS>
struct Operand {
    static constexpr int N = kBlock * BK / 256;      // transfers of a stage
    // bytes, the same for every transfer, `next` elements apart; ROWS = 0: sixteen rows each, off[1] from transfer `full` on, which has rows
    // past the last one
    uint32_t off[ROWS ? 1 : 2];
    uint32_t faddr;
    int64_t next;
    int full, last;
    __device__ __forceinline__ void init(int64_t s_row, int64_t s_k, int rows_left, int lane, uint32_t ring) {
        if constexpr (ROWS == 0) {
            next = 16 * s_row;
            full = rows_left / 16;
            last = (rows_left - 1) / 16;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                off[i] = ((uint32_t)(i ? min(lane >> 2, (rows_left - 1) % 16) : lane >> 2) * (uint32_t)s_row + (uint32_t)k_of(0, lane)) * 4;
        } else {
            next = 4 * s_k;
            off[0] = ((uint32_t)k_of(0, lane) * (uint32_t)s_k + (uint32_t)min((lane & 15) * 4, rows_left - 4)) * 4;
        }
        const int j = lane & 31, half = lane >> 5;
        if constexpr (ROWS == 0) faddr = ring + j * 64 + (((half * 2) ^ ((j >> 1) & 3)) << 4);
        else faddr = ring + half * 8 * kBlock * 4 + j * 8;
    }
    // first k of the stage that this lane's transfer i holds
    static __device__ __forceinline__ int k_of(int i, int lane) {
        if constexpr (ROWS == 0) return ((lane & 3) ^ ((lane >> 3) & 3)) * 4;    // row i * 16 + lane / 4: (row / 2) % 4
        return i * 4 + (lane >> 4);
    }
    // tile row of row j of block b
    static __device__ __forceinline__ int row_of(int b, int j) { return ROWS == 0 ? 32 * b + j : 2 * j + b; }
    __device__ __forceinline__ const char* source(const float* p, int i) const {
        if constexpr (ROWS == 0) return reinterpret_cast<const char*>(p + min(i, last) * next) + (i < full ? off[0] : off[1]);
        else return reinterpret_cast<const char*>(p + i * next) + off[0];
    }
    __device__ __forceinline__ void issue(const float* p, char* stage) const {
#pragma unroll
        for (int i = 0; i < N; ++i) dma(source(p, i), stage + i * 1024);
    }
    // the same for a stage that reaches past the end of K (`left` < 16)
    __device__ __forceinline__ void issue_tail(const float* p, int left, char* stage) const {
        const int lane = lane_again();
#pragma unroll
        for (int i = 0; i < N; ++i)
            dma(k_of(i, lane) < left ? source(p, i) : reinterpret_cast<const char*>(&g_zero_page), stage + i * 1024);
    }
    static __device__ __forceinline__ void dma(const char* p, char* lds_dst) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                         (__attribute__((address_space(3))) void*)lds_dst, 16, 0, 0);
    }
    // this lane's eight k (8 (lane / 32) on) of its row in either block
    struct Raw {
        floatx4 q[4];       // ROWS = 0: two of block 0, two of block 1
        floatx2 p[8];       // ROWS = 1: k by k, both blocks
    };
    __device__ __forceinline__ void read(uint32_t stage, Raw& v) const {
        if constexpr (ROWS == 0) {
            const uint32_t a = faddr + stage;
            v.q[0] = __builtin_bit_cast(floatx4, lds_read_b128<0>(a));
            v.q[1] = __builtin_bit_cast(floatx4, lds_read_b128<0>(a ^ 16));
            v.q[2] = __builtin_bit_cast(floatx4, lds_read_b128<32 * 64>(a));
            v.q[3] = __builtin_bit_cast(floatx4, lds_read_b128<32 * 64>(a ^ 16));
        } else {
            static_for<0, 8>([&](auto ec) {
                constexpr int e = decltype(ec)::value;
                v.p[e] = lds_read_b64<e * kBlock * 4>(faddr + stage);
            });
        }
    }
    // the same from global memory, 16 or 8 bytes at a time; k0: first k of the step, zeros from k on
    static __device__ __forceinline__ void values(const float* p, int64_t s_row, int64_t s_k, int rows_left, int k0, int k, int lane,
                                                  float (&v)[2][8]) {
        const int j = lane & 31, first = k0 + 8 * (lane >> 5);
        if constexpr (ROWS == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int at = first + i % 2 * 4, row = min(32 * (i / 2) + j, rows_left - 1);
                const floatx4 q = *reinterpret_cast<const floatx4*>(p + row * s_row + min(at, k - 4));
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i / 2][i % 2 * 4 + e] = at < k ? q[e] : 0.f;
            }
        } else {
            p += min(2 * j, rows_left - 2);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const floatx2 q = *reinterpret_cast<const floatx2*>(p + min(first + e, k - 1) * s_k);
#pragma unroll
                for (int i = 0; i < 2; ++i) v[i][e] = first + e < k ? q[i] : 0.f;
            }
        }
    }
    // both blocks' pieces, pair by pair: registers of values that are split are free
    static __device__ __forceinline__ void split(const Raw& v, Pieces (&f)[2]) {
        u32x4 h[2], m[2], l[2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int blk = ROWS == 0 ? i / 4 : i % 2, e = ROWS == 0 ? i % 4 : i / 2;
            const floatx2 w = ROWS == 0 ? floatx2{v.q[i / 2][2 * (i % 2)], v.q[i / 2][2 * (i % 2) + 1]} : floatx2{v.p[2 * e][blk], v.p[2 * e + 1][blk]};
            uint32_t ph, pm, pl;
            split_pair(w, kSplitScale, ph, pm, pl);
            h[blk][e] = ph;
            m[blk][e] = pm;
            l[blk][e] = pl;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
            f[i] = {__builtin_bit_cast(bf16x8, h[i]), __builtin_bit_cast(bf16x8, m[i]), __builtin_bit_cast(bf16x8, l[i])};
    }
};

__device__ __forceinline__ float bias_at(const SplitArgs& g, int i) {
    return g.bias_f32 ? reinterpret_cast<const float*>(g.bias)[i] : (float)reinterpret_cast<const _Float16*>(g.bias)[i];
}

// v = alpha * acc + bias, stored to pre; act(v) + residual + beta * C
__device__ __forceinline__ float finish(const SplitArgs& g, float acc, float bias, int64_t off) {
    float v = g.alpha * acc + bias;
    if (g.pre) g.pre[off] = v;
    v = apply_act(g.act, v);
    if (g.residual) v += g.residual[off];
    if (g.beta != 0.f) v += g.beta * g.c[off];
    return v;
}

// The pieces exist from here on: they are not computed where they are used, behind the products that hide them.
__device__ __forceinline__ void keep(Pieces (&p)[2]) {
    asm volatile("" : "+v"(p[0].h), "+v"(p[0].m), "+v"(p[0].l), "+v"(p[1].h), "+v"(p[1].m), "+v"(p[1].l));
}

// A matrix instruction, then what the vector pipe can issue under it
__device__ __forceinline__ void interleave() {
#pragma unroll
    for (int i = 0; i < 12; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 9, 0);
    }
}

// KG: wavefronts, each of which takes every KG-th step of K (16) of the same 64 x 64 tile, with a ring of its own: no barrier in
// the loop. Their sums are added through LDS behind it.
template <int KG, int AROWS, int BROWS>
__global__ __launch_bounds__(kWave * KG, 2) void gemm_f32_split_kernel(const SplitArgs g) {
    constexpr int TB = kBlock, THREADS = kWave * KG;
    constexpr int A_BYTES = kBlock * BK * 4, STAGE = 2 * A_BYTES;
    typedef Operand<AROWS> OA;
    typedef Operand<BROWS> OB;
    constexpr int LPT = OA::N + OB::N;                // transfers per step
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

    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int m0 = tm * TB, n0 = tn * TB;
    char* const ring = lds + wave * kStages * STAGE;
    const uint32_t ring0 = lds_addr(ring);

    floatx16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    OA oa;
    OB ob;
    oa.init(g.sam, g.sak, g.m - m0, lane, ring0);
    ob.init(g.sbn, g.sbk, g.n - n0, lane, ring0 + A_BYTES);
    const int steps = (g.k + BK - 1) / BK, mine = (steps - wave + KG - 1) / KG;
    const float* pa = A + (int64_t)m0 * g.sam + (int64_t)wave * BK * g.sak;
    const float* pb = B + (int64_t)n0 * g.sbn + (int64_t)wave * BK * g.sbk;
    int left = g.k - wave * BK;                       // k from the next transfers' first one on
    auto issue = [&](uint32_t stage) {                // this wavefront's next step
        char* const at = ring + stage;
        if (left >= BK) {
            oa.issue(pa, at);
            ob.issue(pb, at + A_BYTES);
        } else {
            oa.issue_tail(pa, left, at);
            ob.issue_tail(pb, left, at + A_BYTES);
        }
        pa += KG * BK * g.sak;
        pb += KG * BK * g.sbk;
        left -= KG * BK;
    };
    if (mine > 0) {
        typename OA::Raw va;
        typename OB::Raw vb;
        Pieces fa[2][2], fb[2][2];
        typedef std::integral_constant<int, 0> c0;
        typedef std::integral_constant<int, 1> c1;
        typedef std::integral_constant<int, 2> c2;
        floatx16 low[2][2];              // sums of the small products
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) low[i][j][e] = 0.f;
        // Step t, whose pieces are in set CUR, while the values of step t + 1 are split into the other set: A's, read half a step
        // ago, then B's. Half way through every value of step t + 1 is in registers: its stage takes the transfers of step
        // t + 3. LEFT: steps that follow (2 for more).
        auto step = [&](int t, auto cur_c, auto left_c) {
            constexpr int CUR = decltype(cur_c)::value, NXT = CUR ^ 1, LEFT = decltype(left_c)::value;
            const uint32_t here = (uint32_t)((t & 1) * STAGE), other = STAGE - here;
            const Pieces(&a)[2] = fa[CUR];
            const Pieces(&b)[2] = fb[CUR];
            auto products = [&](auto ic) {            // of the two blocks in row I
                constexpr int I = decltype(ic)::value;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    low[I][j] = mfma_small(a[I], b[j], low[I][j]);
                    acc[I][j] = mfma_large(a[I], b[j], acc[I][j]);
                }
            };
            if constexpr (LEFT > 0) {
                wait_lgkm<0>();
                ob.read(other, vb);
                __builtin_amdgcn_sched_barrier(0);
                OA::split(va, fa[NXT]);
            }
            products(c0{});
            if constexpr (LEFT > 0) {
                interleave();
                keep(fa[NXT]);
                __builtin_amdgcn_sched_barrier(0);
                wait_vm_lgkm0<0>();
                if constexpr (LEFT > 1) {
                    oa.read(here, va);
                    if (t + 3 < mine) issue(other);
                }
                __builtin_amdgcn_sched_barrier(0);
                OB::split(vb, fb[NXT]);
            }
            products(c1{});
            if constexpr (LEFT > 0) {
                interleave();
                keep(fb[NXT]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        issue(0);
        if (mine > 1) {
            issue(STAGE);
            wait_vm_lgkm0<LPT>();
        } else {
            wait_vm_lgkm0<0>();
        }
        oa.read(0u, va);
        ob.read(0u, vb);
        wait_lgkm<0>();
        __builtin_amdgcn_sched_barrier(0);
        if (mine > 2) issue(0);
        // the last step works from set 1, so the first one from set mine % 2
        const bool odd = mine & 1;
        if (odd) {
            OA::split(va, fa[1]);
            OB::split(vb, fb[1]);
        } else {
            OA::split(va, fa[0]);
            OB::split(vb, fb[0]);
        }
        if (mine > 1) {
            if (mine > 2) wait_vm_lgkm0<LPT>();
            else wait_vm_lgkm0<0>();
            oa.read(STAGE, va);
            int t = 0;
            if (odd) step(t++, c1{}, c2{});
            for (; t + 2 < mine; t += 2) {
                step(t, c0{}, c2{});
                step(t + 1, c1{}, c2{});
            }
            step(t, c0{}, c1{});
        }
        step(mine - 1, c1{}, c0{});
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] += low[i][j];

        // A value without a split (infinite, NaN, from 2^112 on) makes a sum that is not finite: this wavefront's steps once
        // more, on the fp32 instruction, operands from global memory.
        float bad = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) bad = __builtin_fmaf(acc[i][j][e], 0.f, bad);
        if (__builtin_amdgcn_ballot_w64(bad != 0.f) != 0) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
#pragma unroll 1
            for (int s = wave; s < steps; s += KG) {
                float va[2][8], vb[2][8];
                OA::values(A + (int64_t)m0 * g.sam, g.sam, g.sak, g.m - m0, s * BK, g.k, lane_again(), va);
                OB::values(B + (int64_t)n0 * g.sbn, g.sbn, g.sbk, g.n - n0, s * BK, g.k, lane_again(), vb);
#pragma unroll
                for (int e = 0; e < 8; ++e)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(va[i][e], vb[j][e], acc[i][j], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] *= kSplitBack;
        }
    }
    __syncthreads();                     // the rings are done with
    const int at = lane_again();

    // The wavefronts' sums go through LDS: element e of a block is row (e / 4) * 8 + (lane / 32) * 4 + e % 4, column lane % 32.
    constexpr int PITCH = kBlock + 4;                 // floats; rows stay 16-byte aligned
    static_assert(KG * kBlock * PITCH * 4 <= 160 * 1024, "all partial tiles fit");
    float* const part = reinterpret_cast<float*>(lds);
    {
        float* const own = part + wave * kBlock * PITCH;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = (e >> 2) * 8 + (at >> 5) * 4 + (e & 3);
                float* const row = own + OA::row_of(i, r) * PITCH;
                const float v0 = acc[i][0][e], v1 = acc[i][1][e];
                if constexpr (BROWS) {
                    *reinterpret_cast<floatx2*>(row + 2 * (at & 31)) = floatx2{v0, v1};
                } else {
                    row[at & 31] = v0;
                    row[32 + (at & 31)] = v1;
                }
            }
    }
    __syncthreads();
    constexpr int CPR = kBlock / 4;                   // pieces of four columns per row
    for (int i = wave * kWave + at; i < kBlock * CPR; i += THREADS) {
        const int r = i / CPR, c4 = (i % CPR) * 4;
        const int m = m0 + r, n = n0 + c4;
        if (m >= g.m || n >= g.n) continue;
        floatx4 v = *reinterpret_cast<const floatx4*>(part + r * PITCH + c4);
#pragma unroll
        for (int s = 1; s < KG; ++s) v += *reinterpret_cast<const floatx4*>(part + (s * kBlock + r) * PITCH + c4);
        const int cnt = min(4, g.n - n);
        const int64_t off = coff + (int64_t)m * g.scm + n;
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
}

template <int KG, int AROWS, int BROWS>
int launch(SplitArgs& g, long long batch, hipStream_t st) {
    constexpr int ring = KG * kStages * 2 * kBlock * BK * 4, sums = KG * kBlock * (kBlock + 4) * 4;
    constexpr int lds = ring > sums ? ring : sums;
    g.tiles_m = (g.m + kBlock - 1) / kBlock;
    g.tiles_n = (g.n + kBlock - 1) / kBlock;
    g.total_blocks = (long long)g.tiles_m * g.tiles_n * batch;
    DML_REQUIRE(g.total_blocks <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f32: too many workgroups");
    auto kern = gemm_f32_split_kernel<KG, AROWS, BROWS>;
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) {
        set_error("gemm_f32: cannot reserve %d bytes of LDS: %s", lds, hipGetErrorString(e));
        return (int)e;
    }
    hipLaunchKernelGGL(kern, (unsigned)g.total_blocks, kWave * KG, lds, st, g);
    return launch_status("gemm_f32");
}

template <int AROWS, int BROWS>
int launch_form(SplitArgs& g, int form, long long batch, hipStream_t st) {
    return form == 0 ? launch<8, AROWS, BROWS>(g, batch, st) : launch<4, AROWS, BROWS>(g, batch, st);
}

// ROWS of Operand, -1: 16 bytes at a time do not work. Offsets inside a tile and a step are 32 bits wide.
int operand_rows(const void* p, int64_t rows, int64_t k, int64_t s_row, int64_t s_k, const int64_t* sb, const int64_t* batch) {
    if (!aligned16(p) || 64.0 * s_row + 16.0 * s_k >= 1073741824.0) return -1;
    for (int i = 0; i < 3; ++i)
        if (batch[i] > 1 && sb[i] % 4 != 0) return -1;
    if (s_k == 1 && s_row % 4 == 0 && k % 4 == 0) return 0;
    return s_row == 1 && s_k % 4 == 0 && rows % 4 == 0 ? 1 : -1;
}

thread_local int g_force_tile = -1;   // diagnostic: 0 - 2 = the streamed kernel's tiles, 3 and 4 = the forms here

// -1: the streamed kernel is the faster one. Measured: a step of eight wavefronts on a compute unit takes 1.14 us, whether
// they share a tile or are two workgroups of four (0.61 alone); first loads, the sum through LDS and stores 6.4 us per tile of eight, 7.1 us
// per pair of tiles of four. So one tile per compute unit takes eight (1024 x 768 x 768: 15.9 us, four 16.5, streamed 20; 1024 x
// 768 x 3072 38.6 / 40.1 / 52), more take four (1024 x 3072 x 768: 38.5, eight 45, streamed 51; 4096^3 850 / 880 / 1016). Few
// tiles (512^3: 9.6, streamed 6.0) and short K (512 x 512 x 64, 24 times: 24, streamed 17) stay on the streamed kernel.
// Rows of K that do not start at a multiple of 64 bytes make two requests of each of a step's: 1.4 - 1.55 us for eight wavefronts
// (640 x 472 x 20284, streamed / eight / four, 211 / 253 / 209). Operands of more than the 256 MB of the last-level cache: 1.5 - 2.2 us and
// the streamed kernel a fifth more than it estimates (768 x 36 x 51788, 8 times, 585 / 909 / 806). 680 products of 32 - 4096 rows, K of 16 - 65536:
// none takes more than 1.03 of the streamed kernel's time, 0.91 on average; without these two 1.55, ten more than 1.1.
int choose_form(const dmlhip_gemm_desc* d, long long batch, const void* a, const void* b, int a_rows, int b_rows) {
    const double tiles = (double)ceil_div(d->m, kBlock) * ceil_div(d->n, kBlock) * batch, n = ceil(tiles / kCus);
    auto unaligned = [](const void* p, int rows, int64_t s_row) { return rows == 0 && (s_row % 16 != 0 || reinterpret_cast<uintptr_t>(p) % 64 != 0); };
    double a_bytes = 4.0 * d->m * d->k, b_bytes = 4.0 * d->n * d->k;
    for (int i = 0; i < 3; ++i) {
        if (d->a_stride_batch[i] != 0) a_bytes *= d->batch[i];
        if (d->b_stride_batch[i] != 0) b_bytes *= d->batch[i];
    }
    const bool twice = unaligned(a, a_rows, d->a_stride_m) || unaligned(b, b_rows, d->b_stride_n), memory = a_bytes + b_bytes > 256e6;
    const double step8 = (twice ? 1.5 : 1.14) * (memory ? 1.4 : 1.0);
    const double step4 = twice ? 0.66 * (memory ? 1.5 : 1.0) : 0.61 * (memory ? 1.25 : 1.0);
    const double eight = n * (6.4 + ceil_div(d->k, 8 * BK) * step8), four = ceil(n / 2) * 7.1 + 0.8 + n * ceil_div(d->k, 4 * BK) * step4;
    if (gemm_f32_streamed_us(d, batch) * (memory ? 1.2 : 1.0) <= fmin(eight, four)) return -1;
    return eight <= four ? 0 : 1;
}

}  // namespace
}  // namespace dml

using namespace dml;
extern "C" int dmlhip_gemm_f32(const dmlhip_gemm_desc* d, const void* a, const void* b, void* c, const void* bias,
                               const void* residual, void* pre_out, void* stream) {
    DML_REQUIRE(d, DMLHIP_ERR_NULL, "gemm_f32: NULL descriptor");
    DML_REQUIRE(d->m >= 0 && d->n >= 0 && d->k >= 0, DMLHIP_ERR_SHAPE, "gemm_f32: negative extent");
    DML_REQUIRE(d->m <= 2147483647 / 2 && d->n <= 2147483647 / 2 && d->k <= 2147483647 / 2, DMLHIP_ERR_SHAPE,
                "gemm_f32: extent exceeds 2^30");
    long long batch = 1;
    for (int i = 0; i < 3; ++i) {
        DML_REQUIRE(d->batch[i] >= 0 && d->batch[i] <= 2147483647, DMLHIP_ERR_SHAPE, "gemm_f32: bad batch extent");
        batch *= d->batch[i];
        DML_REQUIRE(batch <= 2147483647LL, DMLHIP_ERR_SHAPE, "gemm_f32: batch too large");
    }
    DML_REQUIRE(d->out_dtype == DMLHIP_F32, DMLHIP_ERR_ENUM, "gemm_f32: out_dtype must be DMLHIP_F32");
    DML_REQUIRE(d->bias_dtype == DMLHIP_F16 || d->bias_dtype == DMLHIP_F32, DMLHIP_ERR_ENUM,
                "gemm_f32: bad bias_dtype");
    DML_REQUIRE(valid_act(d->act), DMLHIP_ERR_ENUM, "gemm_f32: bad act");
    DML_REQUIRE(d->a_stride_m >= 0 && d->a_stride_k >= 0 && d->b_stride_k >= 0 && d->b_stride_n >= 0 &&
                    d->c_stride_m >= 0,
                DMLHIP_ERR_SHAPE, "gemm_f32: negative stride");
    DML_REQUIRE(d->c_stride_m >= d->n || d->m <= 1, DMLHIP_ERR_SHAPE, "gemm_f32: rows of C overlap");
    if (d->m == 0 || d->n == 0 || batch == 0) return 0;
    DML_REQUIRE(c, DMLHIP_ERR_NULL, "gemm_f32: NULL output");
    DML_REQUIRE(d->k == 0 || (a && b), DMLHIP_ERR_NULL, "gemm_f32: NULL operand");

    if (g_force_tile >= 0 && g_force_tile < 3)
        return gemm_f32_streamed(d, a, b, c, bias, residual, pre_out, g_force_tile, batch, (hipStream_t)stream);
    SplitArgs g;
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
    const int ar = operand_rows(a, d->m, d->k, d->a_stride_m, d->a_stride_k, d->a_stride_batch, d->batch);
    const int br = operand_rows(b, d->n, d->k, d->b_stride_n, d->b_stride_k, d->b_stride_batch, d->batch);
    const int form = ar < 0 || br < 0 ? -1 : g_force_tile >= 3 ? g_force_tile - 3 : choose_form(d, batch, a, b, ar, br);
    if (form < 0) return gemm_f32_streamed(d, a, b, c, bias, residual, pre_out, -1, batch, (hipStream_t)stream);
    hipStream_t st = (hipStream_t)stream;
    if (ar == 0) return br == 0 ? launch_form<0, 0>(g, form, batch, st) : launch_form<0, 1>(g, form, batch, st);
    return br == 0 ? launch_form<1, 0>(g, form, batch, st) : launch_form<1, 1>(g, form, batch, st);
}

extern "C" void dmlhip_debug_force_gemm_f32_tile(int tile) { g_force_tile = tile; }
