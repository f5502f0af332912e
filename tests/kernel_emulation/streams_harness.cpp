// Runs one of the kernels that stream their operands into LDS by themselves (compiled for the host against emu.h) on one
// problem; which one is chosen by a macro, since each source has its own names. TEST INFRASTRUCTURE ONLY; built and driven by
// tests/test_kernel_emulation_streams.py.
#include <stdarg.h>
#include <stdio.h>
#include <cmath>

#if defined(EMU_SPLIT)
namespace dml { namespace gemm16 { namespace { alignas(16) char lds[160 * 1024]; } } }
#include "gemm_f16_split_emu.h"
#else
namespace dml { namespace { alignas(16) char lds[160 * 1024]; } }
#if defined(EMU_F32)
#include "gemm_f32_emu.h"
#elif defined(EMU_F32SPLIT)
#include "gemm_f32_split_emu.h"
#elif defined(EMU_DENSE3)
#include "conv_dense3_emu.h"
#elif defined(EMU_DENSE3WS)
#include "conv_dense3_weight_split_emu.h"
#else
#include "conv_dense3_weight_emu.h"
#endif
#endif

namespace dml {
void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    va_end(ap);
    fputc('\n', stderr);
}
int launch_status(const char*) { return 0; }
#if defined(EMU_F32SPLIT)
int gemm_f32_streamed(const dmlhip_gemm_desc*, const void*, const void*, void*, const void*, const void*, void*, int, long long, hipStream_t) { return 0; }
double gemm_f32_streamed_us(const dmlhip_gemm_desc*, long long) { return 0.0; }
#endif
#if defined(EMU_DENSE3) || defined(EMU_DENSE3WS)
void note_conv_form(int) {}
#endif
#if defined(EMU_DENSE3)
// asked by the launch functions only, which are not called here
bool conv_implicit_applicable(const ConvGeom&) { return false; }
bool conv_implicit_bwd_data_applicable(const ConvGeom&) { return false; }
#endif
}  // namespace dml

#if defined(EMU_SPLIT)
using namespace dml::gemm16;

namespace {
struct Call {
    const _Float16 *a, *b;
    void* c;
    GemmArgs g;
};
template <int T, int AK, int BK_, bool KS, bool AS>
void entry(void* p) {
    const Call* c = static_cast<const Call*>(p);
    gemm_f16_split_kernel<T, 2, AK, BK_, EPI_PLAIN, KS, AS>(c->a, c->b, c->c, nullptr, nullptr, nullptr, c->g);
}
template <int T, bool KS, bool AS> emu::kernel_fn pick(int ak, int bk) {
    if (ak) return bk ? entry<T, 1, 1, KS, AS> : entry<T, 1, 0, KS, AS>;
    return bk ? entry<T, 0, 1, KS, AS> : entry<T, 0, 0, KS, AS>;
}
template <bool KS, bool AS> emu::kernel_fn pick_tile(int t, int ak, int bk) {
    return t == 2 ? pick<2, KS, AS>(ak, bk) : pick<1, KS, AS>(ak, bk);
}
}  // namespace

// C[m, n] (fp32) = sum over `pairs` operand pairs; kinds 0 = K contiguous, 1 = rows contiguous; t: tile / 32; asum: row sums
// of A, or NULL
extern "C" int emu_split(int t, int ak, int bk, int m, int n, int k, int pairs, const void* const* a, const void* const* b,
                         float* c, float* asum, unsigned seed, int late) {
    Call call = {};
    GemmArgs& g = call.g;
    g.m = m; g.n = n; g.k = k;
    g.sam = ak ? 1 : k; g.sak = ak ? m : 1;
    g.sbn = bk ? 1 : k; g.sbk = bk ? n : 1;
    g.scm = n;
    g.batch1 = g.batch2 = 1;
    g.alpha = 1.f;
    g.out_f32 = 1;
    g.c_vec = n % 8 == 0;
    g.tiles_m = (m + 32 * t - 1) / (32 * t);
    g.tiles_n = (n + 32 * t - 1) / (32 * t);
    g.total_blocks = (long long)g.tiles_m * g.tiles_n;
    call.a = (const _Float16*)a[0];
    call.b = (const _Float16*)b[0];
    call.c = c;
    if (pairs > 1) {
        g.ksum = 1;
        g.groups = pairs;
        for (int i = 0; i < pairs; ++i) { g.ga[i] = (const _Float16*)a[i]; g.gb[i] = (const _Float16*)b[i]; }
    }
    g.asum = asum;
    g.asum_f32 = 1;
    emu::kernel_fn fn = pairs > 1 ? pick_tile<true, false>(t, ak, bk) : asum ? pick_tile<false, true>(t, ak, bk) : pick_tile<false, false>(t, ak, bk);
    return emu::run_grid(fn, &call, (unsigned)g.total_blocks, kThreads, seed, late, lds);
}

#elif defined(EMU_F32)
using namespace dml;

namespace {
template <int T, int WPG, int KG, int NSTAGE, int AR, int AV, int BR, int BV>
void entry(void* p) { gemm_f32_kernel<T, WPG, KG, NSTAGE, AR, AV, BR, BV>(*static_cast<const GemmArgs32*>(p)); }
template <int AR, int AV, int BR, int BV> emu::kernel_fn pick(int tile) {
    if constexpr (AV == 4 && BV == 4)
        if (tile == 0) return entry<2, 4, 1, 2, AR, AV, BR, BV>;
    return tile <= 1 ? entry<1, 4, 1, 3, AR, AV, BR, BV> : entry<1, 1, 4, 2, AR, AV, BR, BV>;
}
template <int AR, int AV> emu::kernel_fn pick_b(int tile, int mode) {
    switch (mode) {
        case 0: return pick<AR, AV, 0, 4>(tile);
        case 1: return pick<AR, AV, 1, 4>(tile);
        case 2: return pick<AR, AV, 0, 1>(tile);
        default: return pick<AR, AV, 1, 1>(tile);
    }
}
}  // namespace

// kinds 0 = K contiguous, 1 = rows contiguous; the operand modes are the library's own choice
extern "C" int emu_gemm_f32(int tile, int ak, int bk, int m, int n, int k, const float* a, const float* b, float* c, unsigned seed,
                            int late) {
    GemmArgs32 g = {};
    g.a = a; g.b = b; g.c = c;
    g.m = m; g.n = n; g.k = k;
    g.sam = ak ? 1 : k; g.sak = ak ? m : 1;
    g.sbn = bk ? 1 : k; g.sbk = bk ? n : 1;
    g.scm = n;
    g.batch1 = g.batch2 = 1;
    g.alpha = 1.f;
    g.c_vec = n % 4 == 0;
    const int64_t one[3] = {1, 1, 1}, zero[3] = {0, 0, 0};
    const int am = operand_mode32(a, m, k, g.sam, g.sak, zero, one), bm = operand_mode32(b, n, k, g.sbn, g.sbk, zero, one);
    if (tile == 0 && (am > 1 || bm > 1)) tile = 1;
    const int tb = 128 >> tile;
    g.tiles_m = (m + tb - 1) / tb;
    g.tiles_n = (n + tb - 1) / tb;
    g.total_blocks = (long long)g.tiles_m * g.tiles_n;
    emu::kernel_fn fn = am == 0 ? pick_b<0, 4>(tile, bm) : am == 1 ? pick_b<1, 4>(tile, bm) : am == 2 ? pick_b<0, 1>(tile, bm) : pick_b<1, 1>(tile, bm);
    return emu::run_grid(fn, &g, (unsigned)g.total_blocks, 256, seed, late, lds);
}

#elif defined(EMU_F32SPLIT)
using namespace dml;

namespace {
template <int KG, int AR, int BR> void entry(void* p) { gemm_f32_split_kernel<KG, AR, BR>(*static_cast<const SplitArgs*>(p)); }
template <int KG> emu::kernel_fn pick(int ar, int br) {
    if (ar) return br ? entry<KG, 1, 1> : entry<KG, 1, 0>;
    return br ? entry<KG, 0, 1> : entry<KG, 0, 0>;
}
}  // namespace

// K over kg (8 or 4) wavefronts; kinds 0 = K contiguous, 1 = rows contiguous
extern "C" int emu_gemm_f32_split(int kg, int ak, int bk, int m, int n, int k, const float* a, const float* b, float* c, unsigned seed,
                                  int late) {
    SplitArgs g = {};
    g.a = a; g.b = b; g.c = c;
    g.m = m; g.n = n; g.k = k;
    g.sam = ak ? 1 : k; g.sak = ak ? m : 1;
    g.sbn = bk ? 1 : k; g.sbk = bk ? n : 1;
    g.scm = n;
    g.batch1 = g.batch2 = 1;
    g.alpha = 1.f;
    g.c_vec = n % 4 == 0;
    const int64_t one[3] = {1, 1, 1}, zero[3] = {0, 0, 0};
    if (operand_rows(a, m, k, g.sam, g.sak, zero, one) != ak || operand_rows(b, n, k, g.sbn, g.sbk, zero, one) != bk) return 3;
    g.tiles_m = (m + kBlock - 1) / kBlock;
    g.tiles_n = (n + kBlock - 1) / kBlock;
    g.total_blocks = (long long)g.tiles_m * g.tiles_n;
    return emu::run_grid(kg == 8 ? pick<8>(ak, bk) : pick<4>(ak, bk), &g, (unsigned)g.total_blocks, 64 * kg, seed, late, lds);
}

#else
using namespace dml;

static ConvGeom geometry(int n, int c, int h, int w, int m, int s, int p, int d) {
    ConvGeom g = {};
    g.n = n; g.c = c; g.h = h; g.w = w; g.m = m;
    g.kh = g.kw = 3;
    g.sh = g.sw = s; g.ph = g.pw = p; g.dh = g.dw = d;
    g.group = 1;
    g.oh = (h + 2 * p - 2 * d - 1) / s + 1;
    g.ow = (w + 2 * p - 2 * d - 1) / s + 1;
    g.cg = c; g.mg = m;
    return g;
}

#if defined(EMU_DENSE3)
namespace {
template <int TILE, bool FLIP, int VEC, int XVEC>
void entry(void* p) { conv_dense3_f32_kernel<(4 >> TILE), (1 << TILE), FLIP, VEC, XVEC>(*static_cast<const Dense3Args*>(p)); }
template <bool FLIP, int VEC, int XVEC> emu::kernel_fn pick(int tile) {
    return tile == 0 ? entry<0, FLIP, VEC, XVEC> : tile == 1 ? entry<1, FLIP, VEC, XVEC> : entry<2, FLIP, VEC, XVEC>;
}
template <bool FLIP> emu::kernel_fn pick_form(int tile, int vec, int xvec) {
    if (vec == 4) return xvec == 4 ? pick<FLIP, 4, 4>(tile) : pick<FLIP, 4, 1>(tile);
    return xvec == 4 ? pick<FLIP, 1, 4>(tile) : pick<FLIP, 1, 1>(tile);
}
}  // namespace

// the convolution (data = 0: x -> y) or its data gradient (data = 1: x is dY, y is dX). 3: the kernel does not take it
extern "C" int emu_dense3(int tile, int data, int n, int c, int h, int w, int m, int s, int p, int d, const float* x, const float* wt,
                          float* y, unsigned seed, int late) {
    const ConvGeom f = geometry(n, c, h, w, m, s, p, d);
    ConvGeom g = f;
    if (data && !data_gradient_problem(f, &g)) return 3;
    Dense3Plan pl;
    g_force_tile = tile;
    if (!plan_conv_dense3(g, data ? s : 1, data ? s : 1, data != 0, false, x, wt, &pl)) return 3;
    pl.a.x = x; pl.a.w = wt; pl.a.bias = nullptr; pl.a.y = y;
    emu::kernel_fn fn = data ? pick_form<true>(tile, pl.vec, pl.xvec) : pick_form<false>(tile, pl.vec, pl.xvec);
    return emu::run_grid(fn, &pl.a, pl.blocks, 256, seed, late, lds);
}

#else
namespace {
#if defined(EMU_DENSE3WS)
template <int WM, int AV, int XV> void entry(void* p) { conv_dense3_weight_split_kernel<WM, AV, XV>(*static_cast<const WeightArgs*>(p)); }
#else
template <int WM, int AV, int XV> void entry(void* p) { conv_dense3_weight_kernel<WM, AV, XV>(*static_cast<const WeightArgs*>(p)); }
#endif
template <int WM> emu::kernel_fn pick(int av, int xv) {
    if (av == 4) return xv == 4 ? entry<WM, 4, 4> : entry<WM, 4, 1>;
    return xv == 4 ? entry<WM, 1, 4> : entry<WM, 1, 1>;
}
}  // namespace

// part[ranges][m * c * 9], in chunks of at most `rows` output rows. 3: the kernel does not take it
extern "C" int emu_dense3_weight(int n, int c, int h, int w, int m, int s, int p, int d, int ranges, int rows, const float* x,
                                 const float* dy, float* part, unsigned seed, int late) {
    const ConvGeom g = geometry(n, c, h, w, m, s, p, d);
    WeightPlan pl;
    unsigned blocks;
    int av, xv;
    if (!plan_weight(g, x, dy, &pl, &blocks, &av, &xv)) return 3;
    const int mb = m > 32 ? 64 : 32;
    if (!lay_out(g, rows < g.oh ? rows : g.oh, av, xv, mb, &pl)) return 3;
    pl.a.x = x; pl.a.dy = dy; pl.a.part = part;
    pl.a.ranges = ranges;
    return emu::run_grid(m > 32 ? pick<2>(av, xv) : pick<1>(av, xv), &pl.a, (unsigned)(ranges * pl.a.tiles_m * pl.a.tiles_c), kThreads, seed, late, lds);
}
#endif
#endif
