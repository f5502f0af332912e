// Depthwise 3 x 3 and 5 x 5 convolutions, fp32, stride 1, no dilation, output as large as the input: forward, data gradient
// (the same with the taps reversed) and weight gradient.
//
// What bounds them: memory, if enough of it is in flight. A thread owns four columns of a strip of rows: it issues all loads
// of the strip at once - per input row one of 16 bytes and the K - 1 neighbours, which the L1 has - keeps the rows in
// registers, and every input value is used for all taps it reaches. No LDS, no barrier; threads are counted through all
// planes, so that small planes fill wavefronts like large ones. Where a row is no multiple of four columns, the last four
// overlap the ones before (the same values are computed and written twice), and 16-byte accesses are 4-byte aligned
// (4-byte loads instead, every fourth column per lane, took twice as long as aligned ones: 41 us at 55 x 55).
// Measured, us forward / data gradient / weight gradient (with its sum over the images), before (an LDS tile per plane; a
// thread per cell with 4-byte loads; a workgroup per plane) and now: 32 x 144 planes of 56 x 56 34 / 60 / 51 and
// 22 / 22 / 31 (58 MB in, 58 MB out: a copy of that size in memory takes 25, these are partly in the last-level cache),
// 55 x 55 41 / 60 / 47 and 20 / 20 / 32, 32 x 480 of 14 x 14 35 / 16 / 26 and 7 / 7 / 13, 5 x 5 on 32 x 240 of 28 x 28
// 37 / 55 / 116 and 18 / 18 / 31.
#include "common.h"
#include "conv_geom.h"

#include <type_traits>

namespace dml {
namespace {

struct PlaneArgs {
    const float* x;
    const float* w;          // forward / data gradient
    const float* bias;
    const float* dy;         // weight gradient
    float* out;
    int c, h, wd;
    int cw, cells;           // column groups of a row, (strip, column group) cells of a plane
    uint32_t total;          // cells, or planes, of all images and channels
    int act;
};

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
template <bool VEC> struct Four { typedef floatx4 type; };      // VEC: 16-byte aligned
template <> struct Four<false> { typedef floatx4u type; };

template <int K> constexpr int strip_rows() { return K == 3 ? 7 : 4; }

// Rows y0 - K/2 .. of the four columns from c0, with K / 2 columns either side; zeros outside the plane.
template <int K, int ROWS, bool VEC>
__device__ __forceinline__ void load_rows(const float* __restrict__ plane, int h, int wd, int y0, int c0, float (&v)[ROWS][K + 3]) {
    constexpr int P = K / 2;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const int iy = y0 - P + r;
        const bool rok = iy >= 0 && iy < h;
        const float* row = plane + (rok ? iy : 0) * wd;
        const typename Four<VEC>::type m = *reinterpret_cast<const typename Four<VEC>::type*>(row + c0);
#pragma unroll
        for (int j = 0; j < K + 3; ++j) {
            const int ix = c0 - P + j;
            if (j < P || j >= P + 4) {
                const bool ok = rok && ix >= 0 && ix < wd;
                v[r][j] = row[ok ? ix : 0];
                v[r][j] = ok ? v[r][j] : 0.f;
            } else {
                v[r][j] = rok ? m[j - P] : 0.f;
            }
        }
    }
}

template <int K, bool VEC, bool FLIP>
__global__ __launch_bounds__(256) void depthwise_same_kernel(const PlaneArgs g) {
    constexpr int R = strip_rows<K>();
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= g.total) return;
    const uint32_t plane = idx / (uint32_t)g.cells;
    const int cell = (int)(idx - plane * (uint32_t)g.cells), strip = cell / g.cw;
    const int y0 = strip * R, c0 = min(4 * (cell - strip * g.cw), g.wd - 4);
    const int ch = (int)(plane % (uint32_t)g.c);
    float v[R + K - 1][K + 3];
    load_rows<K, R + K - 1, VEC>(g.x + (size_t)plane * g.h * g.wd, g.h, g.wd, y0, c0, v);
    float wk[K * K];
#pragma unroll
    for (int i = 0; i < K * K; ++i) wk[i] = g.w[ch * K * K + (FLIP ? K * K - 1 - i : i)];
    const float bias = !FLIP && g.bias ? g.bias[ch] : 0.f;
    float* out = g.out + (size_t)plane * g.h * g.wd + (size_t)y0 * g.wd + c0;
    auto store = [&](auto actc) {
        constexpr int ACT = decltype(actc)::value;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (y0 + r >= g.h) break;
            typename Four<VEC>::type o;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float acc = bias;
#pragma unroll
                for (int hy = 0; hy < K; ++hy)
#pragma unroll
                    for (int hx = 0; hx < K; ++hx) acc += wk[hy * K + hx] * v[r + hy][j + hx];
                o[j] = apply_act(ACT, acc);
            }
            *reinterpret_cast<typename Four<VEC>::type*>(out + r * g.wd) = o;
        }
    };
    switch (FLIP ? DMLHIP_ACT_NONE : g.act) {
        case DMLHIP_ACT_SWISH: store(std::integral_constant<int, DMLHIP_ACT_SWISH>{}); break;
        case DMLHIP_ACT_SIGMOID: store(std::integral_constant<int, DMLHIP_ACT_SIGMOID>{}); break;
        case DMLHIP_ACT_RELU: store(std::integral_constant<int, DMLHIP_ACT_RELU>{}); break;
        case DMLHIP_ACT_GELU: store(std::integral_constant<int, DMLHIP_ACT_GELU>{}); break;
        default: store(std::integral_constant<int, DMLHIP_ACT_NONE>{}); break;
    }
}

// G lanes share a plane; K * K sums per lane over its cells, added across the group. out: [plane][K * K].
template <int K, bool VEC, int G>
__global__ __launch_bounds__(256) void depthwise_same_weight_kernel(const PlaneArgs g) {
    constexpr int R = strip_rows<K>(), P = K / 2;
    const uint32_t plane = (blockIdx.x * 256u + threadIdx.x) / G;
    const int lane = (int)threadIdx.x % G;
    const bool live = plane < g.total;
    const size_t base = (size_t)(live ? plane : 0) * g.h * g.wd;
    // four rows' products per tap are summed on their own: one chain over all cells of a lane was 2.7 times as far from the
    // exact sum as the general kernel's 256 shorter ones (8 planes of 448 x 448: 1.3e-7 of it)
    float total[K * K];
#pragma unroll
    for (int i = 0; i < K * K; ++i) total[i] = 0.f;
    for (int cell = lane; live && cell < g.cells; cell += G) {
        const int strip = cell / g.cw, first = 4 * (cell - strip * g.cw), y0 = strip * R;
        const int c0 = min(first, g.wd - 4);
        float v[R + K - 1][K + 3], d[R][4], acc[K * K];
        load_rows<K, R + K - 1, VEC>(g.x + base, g.h, g.wd, y0, c0, v);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool rok = y0 + r < g.h;
            const float* row = g.dy + base + (size_t)(rok ? y0 + r : 0) * g.wd;
            const typename Four<VEC>::type m = *reinterpret_cast<const typename Four<VEC>::type*>(row + c0);
#pragma unroll
            for (int j = 0; j < 4; ++j) d[r][j] = rok ? m[j] : 0.f;
        }
        // Products with a pixel outside either plane, or with a column that the thread before has added, are left out and not
        // multiplied by zero: the other factor may be infinite.
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r % 4 == 0) {
#pragma unroll
                for (int i = 0; i < K * K; ++i) acc[i] = 0.f;
            }
#pragma unroll
            for (int hy = 0; hy < K; ++hy) {
                const int iy = y0 + r + hy - P;
                const bool rows = y0 + r < g.h && iy >= 0 && iy < g.h;
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int hx = 0; hx < K; ++hx) {
                        const int ix = c0 + j + hx - P;
                        const bool edge = j + hx < P || j + hx >= P + 4;
                        float& sum = acc[hy * K + hx];
                        if (VEC && hy == P && !edge) {        // either both rows exist or both factors are zero
                            sum += d[r][j] * v[r + hy][j + hx];
                        } else {
                            const bool ok = rows && (!edge || (ix >= 0 && ix < g.wd)) && (VEC || c0 + j >= first);
                            sum += ok ? d[r][j] * v[r + hy][j + hx] : 0.f;
                        }
                    }
            }
            if (r % 4 == 3 || r == R - 1) {
#pragma unroll
                for (int i = 0; i < K * K; ++i) total[i] += acc[i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < K * K; ++i)
#pragma unroll
        for (int s = 1; s < G; s *= 2) total[i] += __shfl_xor(total[i], s);
    if (live && lane == 0) {
#pragma unroll
        for (int i = 0; i < K * K; ++i) g.out[(size_t)plane * K * K + i] = total[i];
    }
}

bool same_size(int kh, int kw, int sh, int sw, int ph, int pw, int dh, int dw, int h, int w, int oh, int ow) {
    return kh == kw && (kh == 3 || kh == 5) && sh == 1 && sw == 1 && dh == 1 && dw == 1 && ph == kh / 2 && pw == kw / 2 &&
           oh == h && ow == w && w >= 4 && (int64_t)h * w <= (1 << 28);
}

template <int K>
void fill(PlaneArgs& a, int c, int h, int wd) {
    a.c = c; a.h = h; a.wd = wd;
    a.cw = (wd + 3) / 4;
    a.cells = a.cw * ((h + strip_rows<K>() - 1) / strip_rows<K>());
}

template <int K, bool FLIP>
int launch_same(PlaneArgs a, int64_t planes, int h, int wd, bool vec, hipStream_t st, const char* what) {
    fill<K>(a, a.c, h, wd);
    a.total = (uint32_t)(planes * a.cells);
    const unsigned blocks = (unsigned)ceil_div(planes * a.cells, (int64_t)256);
    if (vec) hipLaunchKernelGGL((depthwise_same_kernel<K, true, FLIP>), blocks, 256, 0, st, a);
    else hipLaunchKernelGGL((depthwise_same_kernel<K, false, FLIP>), blocks, 256, 0, st, a);
    return launch_status(what);
}

template <int K, bool VEC>
int launch_same_weight(PlaneArgs a, int64_t planes, int h, int wd, hipStream_t st) {
    fill<K>(a, a.c, h, wd);
    a.total = (uint32_t)planes;
    const int lanes = a.cells > 32 ? 64 : a.cells > 16 ? 32 : a.cells > 8 ? 16 : 8;
    const unsigned blocks = (unsigned)ceil_div(planes * lanes, (int64_t)256);
#define DML_DWSW(G) \
    if (lanes == G) hipLaunchKernelGGL((depthwise_same_weight_kernel<K, VEC, G>), blocks, 256, 0, st, a);
    DML_DWSW(8) DML_DWSW(16) DML_DWSW(32) DML_DWSW(64)
#undef DML_DWSW
    return launch_status("conv2d_backward_weight(depthwise)");
}

// Whether the kernels above are faster than those that cover the other depthwise convolutions too (a plane's tile in LDS; a
// thread per four outputs; a workgroup per plane), from 1200 problems of 8 - 6144 planes of 4 x 4 to 448 x 448 timed on both,
// us there / here. Few small planes are a matter of latency alone, and a strip's loads take longer than a tile's: forward
// 256 planes of 4 x 4 2.8 / 5.2, of 12 x 12 3.4 / 4.7, of 28 x 28 4.6 / 4.6, of 33 x 33 6.7 / 4.6; data gradient 256 planes of
// 28 x 28 3.2 / 3.8, of 40 x 40 4.8 / 3.9. The more planes, the smaller they may be (forward, 14 x 14: 512 4.5 / 4.7,
// 1536 6.7 / 4.8). vec: rows in 16-byte pieces, which spread planes below 17 columns over a quarter of the lanes.
// A single row fills a seventh of a strip: data gradient of 5120 planes of 1 x 1000 11.1 / 15.7, of 2 x 512 17.6 / 11.3.
bool same_faster(int64_t planes, int h, int64_t hw, int k, bool vec, bool data) {
    if (data && h == 1 && hw >= 512) return false;
    if (hw > (data ? 1024 : 784)) return true;      // forward, 8 planes of 29 x 29 5.8 / 4.2
    if (hw >= 784) return planes >= 384;
    const bool wide = k == 5 && !data;           // forward 5 x 5: a sixth more before a strip's loads are paid for
    if (hw > 256) return planes >= (wide ? 768 : 512);
    if (vec) return planes >= (hw > 64 ? 1408 : wide ? 3584 : 2816);
    if (hw > 49) return planes >= 1024;
    return planes >= (wide ? 1280 : 1024) || (data && k == 5);      // 256 planes of 5 x 5: 4.4 / 4.0
}

// The same for the weight gradient, where a plane has at most one wavefront here and four there: 3 x 3 on 96 planes of
// 14 x 14 2.7 / 6.3, 768 of 56 x 56 13.0 / 11.9, 480 of 111 x 111 32.3 / 33.0, 4096 of 14 x 14 10.4 / 9.2, 5120 of 3 x 301 23.8 / 26.6;
// 5 x 5 on 512 planes of 12 x 12 7.8 / 9.1, of 24 x 24 12.5 / 9.7, 96 of 112 x 112 116 / 56. Few planes under 5 x 5 wait for every pass of
// their wavefront, full or not: 29 x 29 is one full pass, 11.4 / 8.9, 60 x 33 three that are two thirds full, 21.0 / 28.9.
template <int K> bool full_passes(int h, int wd, bool vec) {
    const int64_t cells = (int64_t)((wd + 3) / 4) * ((h + strip_rows<K>() - 1) / strip_rows<K>());
    const int64_t held = ceil_div(cells, (int64_t)64) * 64 * 4 * strip_rows<K>();
    return (int64_t)h * wd * 100 >= held * (vec ? 45 : 75);
}
bool same_weight_faster(int64_t planes, int h, int wd, int k, bool vec) {
    const int64_t hw = (int64_t)h * wd;
    if (hw <= 16) return planes >= (k == 3 ? 6144 : 3072);
    if (k == 5) {
        if (planes >= (vec ? 1536 : 2048)) return true;
        return hw >= (vec ? (planes >= 384 ? 400 : 576) : 784) && (planes >= (vec ? 1024 : 512) || full_passes<5>(h, wd, vec));
    }
    if (hw >= 512 && h <= (vec ? 1 : 3)) return false;
    if (!vec) return planes >= 4096 || (planes >= 2048 && hw >= 1024) || (planes >= 1024 && hw >= 8192);
    return planes >= 3072 || planes * hw >= 2000000 || hw >= 40000 || (planes >= 768 && planes * hw >= 800000);
}

thread_local int g_force_same = -1;   // diagnostic: 0 = never, 1 = wherever they apply

// every thread index and element offset fits 32 bits
bool in_range(int64_t planes, int h, int wd) { return planes * h * wd < (1LL << 31) && planes * ((wd + 3) / 4) * ((h + 3) / 4) < (1LL << 31) && planes < (1LL << 25); }

}  // namespace

static bool vec_rows(const ConvGeom& g, const void* a, const void* b) { return g.w % 4 == 0 && aligned16(a) && aligned16(b); }

// a group == c == m convolution of n images
bool depthwise_same_applicable(const ConvGeom& g) {
    return g.group == g.c && g.m == g.c && in_range((int64_t)g.n * g.c, g.h, g.w) &&
           same_size(g.kh, g.kw, g.sh, g.sw, g.ph, g.pw, g.dh, g.dw, g.h, g.w, g.oh, g.ow);
}

bool depthwise_same_faster(const ConvGeom& g, const void* in, const void* out, bool data) {
    if (g_force_same >= 0) return g_force_same != 0;
    return same_faster((int64_t)g.n * g.c, g.h, (int64_t)g.h * g.w, g.kh, vec_rows(g, in, out), data);
}

bool depthwise_same_weight_faster(const ConvGeom& g, const void* x, const void* dy) {
    if (g_force_same >= 0) return g_force_same != 0;
    return same_weight_faster((int64_t)g.n * g.c, g.h, g.w, g.kh, vec_rows(g, x, dy));
}

int launch_depthwise_same(const ConvGeom& g, const float* x, const float* w, const float* bias, float* y, hipStream_t st) {
    PlaneArgs a = {};
    a.x = x; a.w = w; a.bias = bias; a.out = y; a.c = g.c; a.act = g.act;
    const bool vec = vec_rows(g, x, y);
    const int64_t planes = (int64_t)g.n * g.c;
    return g.kh == 3 ? launch_same<3, false>(a, planes, g.h, g.w, vec, st, "conv2d(depthwise)")
                     : launch_same<5, false>(a, planes, g.h, g.w, vec, st, "conv2d(depthwise)");
}

int launch_depthwise_same_bwd_data(const ConvGeom& g, const float* dy, const float* w, float* dx, hipStream_t st) {
    PlaneArgs a = {};
    a.x = dy; a.w = w; a.out = dx; a.c = g.c;
    const bool vec = vec_rows(g, dy, dx);
    const int64_t planes = (int64_t)g.n * g.c;
    return g.kh == 3 ? launch_same<3, true>(a, planes, g.h, g.w, vec, st, "conv2d_backward_data(depthwise)")
                     : launch_same<5, true>(a, planes, g.h, g.w, vec, st, "conv2d_backward_data(depthwise)");
}

int launch_depthwise_same_bwd_weight(const ConvGeom& g, const float* x, const float* dy, float* part, hipStream_t st) {
    PlaneArgs a = {};
    a.x = x; a.dy = dy; a.out = part; a.c = g.c;
    const bool vec = vec_rows(g, x, dy);
    const int64_t planes = (int64_t)g.n * g.c;
    if (g.kh == 3) return vec ? launch_same_weight<3, true>(a, planes, g.h, g.w, st) : launch_same_weight<3, false>(a, planes, g.h, g.w, st);
    return vec ? launch_same_weight<5, true>(a, planes, g.h, g.w, st) : launch_same_weight<5, false>(a, planes, g.h, g.w, st);
}

}  // namespace dml

extern "C" void dmlhip_debug_force_conv_depthwise(int strips) { dml::g_force_same = strips; }
