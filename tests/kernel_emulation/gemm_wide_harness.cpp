// Runs the fp16 GEMM whose workgroups stay for several tiles (daceml_amd/csrc/gemm_f16_wide.h, compiled for the host against emu.h)
// on one problem. TEST INFRASTRUCTURE ONLY; built and driven by tests/test_kernel_emulation_gemm_wide.py, which puts emu:: calls in
// the place of the kernel's inline assembly.
#include <stdarg.h>
#include <stdio.h>

#include "common.h"

namespace emu {

// a buffer's descriptor: transfers from beyond its end are counted and bring zeros
struct rsrc { const char* base; uint32_t bytes; };
static int g_outside = 0;
static const char kZeros[16] = {};

inline rsrc make_rsrc(void* p, int, int bytes, int) { return {(const char*)p, (uint32_t)bytes}; }

inline void buffer_load_lds(rsrc r, void* lds, int size, int lane_offset, int offset, int, int) {
    const uint64_t at = (uint64_t)(uint32_t)lane_offset + (uint32_t)offset;
    const bool inside = at + size <= r.bytes;
    g_outside += !inside;
    dma_issue(inside ? r.base + at : kZeros, (uint32_t)((const char*)lds - g_lds) + size * (thread_idx().x & 63), size);
}

// D = C + A B, 16 x 16 x 32: lane l holds row l % 16 of A and column l % 16 of B for k = 8 (l / 16) .. + 7, and of C / D column
// l % 16, rows 4 (l / 16) + e.
inline dml::floatx4 mfma_16x16x32(h8 a, h8 b, dml::floatx4 c) {
    struct Ops { h8 a, b; } mine = {a, b};
    const Ops* all = static_cast<const Ops*>(wave_exchange(&mine, sizeof(mine)));
    const int lane = thread_idx().x & 63, col = lane & 15;
    for (int e = 0; e < 4; ++e) {
        const int row = 4 * (lane / 16) + e;
        float acc = 0.f;
        for (int k = 0; k < 32; ++k) acc += (float)all[row + 16 * (k / 8)].a[k % 8] * (float)all[col + 16 * (k / 8)].b[k % 8];
        c[e] += acc;
    }
    return c;
}

// a row of sixteen lanes turned by eight; `old` in the banks of four lanes that the mask leaves out
inline uint32_t row_turn(uint32_t old, uint32_t v, int banks) {
    const uint32_t* all = static_cast<const uint32_t*>(wave_exchange(&v, sizeof(v)));
    const int lane = thread_idx().x & 63;
    const uint32_t other = all[lane ^ 8];
    return banks >> (lane % 16 / 4) & 1 ? other : old;
}

inline float shfl_xor(float v, int mask) {
    const float* all = static_cast<const float*>(wave_exchange(&v, sizeof(v)));
    return all[(thread_idx().x & 63) ^ mask];
}

}  // namespace emu

#define __amdgpu_buffer_rsrc_t emu::rsrc
#define __builtin_amdgcn_make_buffer_rsrc emu::make_rsrc
#define __builtin_amdgcn_raw_ptr_buffer_load_lds emu::buffer_load_lds
#define __shfl_xor emu::shfl_xor

#include "gemm_f16_wide.h"

namespace dml {
void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    va_end(ap);
    fputc('\n', stderr);
}
int launch_status(const char*) { return 0; }

namespace gemm16 {
namespace {

alignas(16) char lds[160 * 1024];   // the array the kernel declares `extern __shared__`

struct Call {
    const _Float16 *a, *b;
    void* c;
    const void *bias, *res;
    GemmArgs g;
};

template <int T, int AK, int BKD, int EPI, bool KSUM, bool SLICED>
void entry(void* p) {
    const Call* c = static_cast<const Call*>(p);
    gemm_f16_wide_kernel<T, AK, BKD, EPI, KSUM, SLICED>(c->a, c->b, c->c, c->bias, c->res, c->g);
}

struct Built { int t, ak, bk, epi; bool ksum, sliced; emu::kernel_fn fn; };
#define BUILT(T, AK, BKD, EPI, KSUM, SLICED) {T, AK, BKD, EPI, KSUM, SLICED, entry<T, AK, BKD, EPI, KSUM, SLICED>}
const Built kBuilt[] = {   // EMU_SET: a few in each of several builds, which compile side by side
#if EMU_SET == 0
    BUILT(4, 0, 1, EPI_PLAIN, true, false),
#elif EMU_SET == 1
    BUILT(4, 0, 0, EPI_GENERAL, false, false), BUILT(8, 0, 0, EPI_PLAIN, false, false),
#elif EMU_SET == 2
    BUILT(8, 1, 0, EPI_PLAIN, false, false),
#elif EMU_SET == 3
    BUILT(8, 1, 1, EPI_GENERAL, false, false),
#elif EMU_SET == 4
    BUILT(8, 0, 1, EPI_PLAIN, true, false),
#elif EMU_SET == 5
    BUILT(8, 1, 1, EPI_PLAIN, false, true),
#elif EMU_SET == 6
    BUILT(8, 1, 0, EPI_PLAIN, false, true),
#endif
};

}  // namespace
}  // namespace gemm16
}  // namespace dml

using namespace dml::gemm16;

// C (fp32 or fp16, [m, n] dense) = sum over `pairs` operand pairs of A_i B_i (+ column bias in fp32, + residual of C's type), on
// `blocks` workgroups. akind / bkind as in emu_gemm. slices > 0: partial results [slices][m][n] in fp32, and partial row sums of A
// in `sums` [slices][columns of tiles][2][m]. Returns 0, 1 on a deadlock, 2 for a combination that is not built, 3 where a transfer
// read beyond its operand.
extern "C" int emu_gemm_wide(int t, int akind, int bkind, int m, int n, int k, int pairs, int slices, int out_f32, int blocks,
                             const void* const* a, const void* const* b, void* c, const void* bias, const void* res, float* sums,
                             unsigned seed, int late_dma) {
    Call call = {};
    GemmArgs& g = call.g;
    g.m = m; g.n = n; g.k = k;
    g.sam = akind ? 1 : k; g.sak = akind ? m : 1;
    g.sbn = bkind ? 1 : k; g.sbk = bkind ? n : 1;
    g.scm = n;
    g.batch1 = g.batch2 = 1;
    g.alpha = 1.f;
    g.out_f32 = out_f32;
    g.bias_f32 = 1;
    g.c_vec = 1;
    const int tile = 32 * t;
    g.tiles_m = (m + tile - 1) / tile;
    g.tiles_n = (n + tile - 1) / tile;
    g.total_blocks = (long long)g.tiles_m * g.tiles_n * (slices ? slices : 1);
    call.a = (const _Float16*)a[0];
    call.b = (const _Float16*)b[0];
    call.c = c;
    call.bias = bias;
    call.res = res;
    if (pairs > 1) {
        g.ksum = 1;
        g.groups = pairs;
        for (int i = 0; i < pairs; ++i) { g.ga[i] = (const _Float16*)a[i]; g.gb[i] = (const _Float16*)b[i]; }
    }
    if (slices) {
        g.groups = 1;
        g.batch1 = slices;
        g.scb[1] = (int64_t)m * n;
        g.ga[0] = call.a; g.gb[0] = call.b; g.gc[0] = c;
        g.asum = sums;
    }
    const int epi = res ? EPI_GENERAL : EPI_PLAIN;
    for (const Built& built : kBuilt)
        if (built.t == t && built.ak == akind && built.bk == bkind && built.epi == epi && built.ksum == (pairs > 1) && built.sliced == (slices > 0)) {
            emu::g_outside = 0;
            const int e = emu::run_grid(built.fn, &call, blocks < g.total_blocks ? blocks : (unsigned)g.total_blocks, kThreads, seed, late_dma, lds);
            return e ? e : emu::g_outside ? 3 : 0;
        }
    return 2;
}
