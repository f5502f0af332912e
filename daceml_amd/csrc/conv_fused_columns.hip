// Pointwise (1x1) convolution + activation followed by a 3x3 depthwise convolution + activation without the expanded tensor
// anywhere but in registers: conv_fused.hip's problem for few input channels and wide images.
//
// With the pixels as rows of the fp32 matrix instruction and 32 expanded channels as its columns a lane receives sixteen
// results of one channel. Which pixel is loaded into which row is free: each half of the wavefront is given sixteen consecutive
// columns of one image row, the 14 of its own and one of padding or of the neighbour on each side. The 3x3 stencil then needs
// nothing from another lane: its sums (14 per row and lane at stride 1, 7 at stride 2) stay in registers while the wavefront moves
// down the image, its nine weights are nine registers, and no two wavefronts wait for each other. The results cross LDS once,
// within the wavefront, so that stores run along the rows.
//
// Bound by vector issue plus the matrix pipe, which take turns with fp32 operands: per row of sixteen columns 8 MFMAs of 64 clocks
// for every 16 input channels, 16 + 7 (14) activations, an exponential and a reciprocal each, and 63 / 2 (126) multiply-adds.
// The kernels that keep expanded rows in LDS issue as much, and wait at a barrier per row for the loads of the next one.
// [96,32,112,112] -> 192 channels, swish / swish: stride 2 338 -> 232 us,
// stride 1 780 -> 484 us (1.08 GB of X and results); [24,16,112,112] -> 96, stride 2 42 -> 27, stride 1 102 -> 45.
// Every sum is added in the order of the other kernels: the results are the same bits.
//
// POOL: the results' mean over an image and channel too (the squeeze-excite gate's input), from the registers they are stored
// from: a lane adds its row's results to a sum of its own, and a launch behind adds up the wavefronts' sums. Sums of rows are added
// in fp64: a row is few values, but there are many rows and wavefronts (fp32 throughout 7.0e-8 from the mean in fp64, the
// separate kernel 5.4e-8, so 2.7e-8). This kernel and the separate mean / with the mean, us: [96,32,112,112] -> 192, stride 2
// 258 / 228, stride 1 667 / 485; [96,48,56,56] -> 288 241 / 190; [24,16,112,112] -> 96, stride 2 34.1 / 29.0; one image 9.8 / 9.1.
#include "common.h"
#include "conv_geom.h"

namespace dml {
namespace {

constexpr int kColWaves = 4;
constexpr int kColCB = 32;       // expanded channels per wavefront
constexpr int kColMaxCin = 48;
constexpr int kColFresh = 14;    // columns of a unit that the next unit does not read as its own
constexpr int kColPitch = 29;    // floats per channel in the exchange buffer: odd

constexpr int kBufferFlags = 0x00020000;   // raw buffer, 32-bit data

struct ColArgs {
    int cmid, h, w, oh, ow, act1, act2;
    int seg_rows, cunits, units;     // output rows of a unit; units along a row; units of an image
    uint32_t pairs, cblocks, total;  // wavefronts per image and channel block; channel blocks; wavefronts
    uint32_t blocks;
    float* sums;                     // POOL: [image][pair][expanded channel]
};

__device__ __forceinline__ float col_swish(float v) { return v * sigmoid_epilogue_f(v); }

// SWISH: known when compiling (a run-time choice costs a copy of every value where its branches meet)
template <bool SWISH, int N>
__device__ __forceinline__ void col_activate(float (&v)[N], int act) {
    if (SWISH || act == DMLHIP_ACT_SWISH) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = col_swish(v[i]);
    } else if (act == DMLHIP_ACT_RELU) {
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = fmaxf(v[i], 0.f);
    }
}

template <int CHUNKS, int STRIDE, bool SWISH, bool POOL>
__global__ __launch_bounds__(kColWaves * 64, 3) void expand_depthwise_columns_kernel(const float* __restrict__ x,
                                                                                  const float* __restrict__ we,
                                                                                  const float* __restrict__ be,
                                                                                  const float* __restrict__ wd,
                                                                                  const float* __restrict__ bd,
                                                                                  float* __restrict__ y, const ColArgs a) {
    constexpr int kCin = CHUNKS * 16;
    constexpr int kOut = kColFresh / STRIDE;               // output columns of a unit
    __shared__ float exchange[kColWaves][kColCB * kColPitch];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 31, hh = lane >> 5;

    // the channel blocks of one pair of units read the same pixels: consecutive workgroup numbers go to different XCDs, so
    // renumber to keep them in one L2
    uint32_t bid = blockIdx.x;
    if (a.blocks % 8u == 0) bid = (bid % 8u) * (a.blocks / 8u) + bid / 8u;
    const uint32_t task = bid * kColWaves + (uint32_t)wave;
    if (task >= a.total) return;
    const int c0 = (int)(task % a.cblocks) * kColCB;
    const uint32_t rest = task / a.cblocks;
    const int pair = (int)(rest % a.pairs);
    const int n = (int)(rest / a.pairs);
    const int u0 = 2 * pair, u1 = min(u0 + 1, a.units - 1);
    const bool second = u0 + 1 < a.units;                  // an odd number of units: the last one twice, stored once
    const int seg0 = u0 / a.cunits, seg1 = u1 / a.cunits;
    const int cu0 = u0 - seg0 * a.cunits, cu1 = u1 - seg1 * a.cunits;

    // ---- the lane that loads row m of the matrix operand: unit (m / 4) % 2, column 4 (m / 8) + m % 4 of its sixteen
    const int plane = a.h * a.w;
    const bool lhalf = (j >> 2) & 1;
    const int lcol = min(max((lhalf ? cu1 : cu0) * kColFresh - 1 + 4 * (j >> 3) + (j & 3), 0), a.w - 1);
    int lrow = (lhalf ? seg1 : seg0) * a.seg_rows * STRIDE - 1;
    const uint32_t lbase = (uint32_t)(hh * plane + lcol);
    // uniform offsets (the channel) ride in the instruction: no address arithmetic per load or store
    const auto xbuf = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)n * kCin * plane), 0, kCin * plane * 4, kBufferFlags);
    float px[CHUNKS * 8], wr[CHUNKS * 8];
    auto load_row = [&]() {
        const uint32_t off = (lbase + (uint32_t)(min(max(lrow, 0), a.h - 1) * a.w)) * 4u;
#pragma unroll
        for (int s = 0; s < CHUNKS * 8; ++s)
            px[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xbuf, off, 2 * s * plane * 4, 0));
        ++lrow;
    };
    load_row();

    // ---- the lane that holds channel c0 + j of unit hh
#pragma unroll
    for (int s = 0; s < CHUNKS * 8; ++s) wr[s] = we[(size_t)(c0 + j) * kCin + 2 * s + hh];
    float taps[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) taps[t] = wd[(size_t)(c0 + j) * 9 + t];
    const float bias1 = be ? be[c0 + j] : 0.f, bias2 = bd ? bd[c0 + j] : 0.f;
    const int col = (hh ? cu1 : cu0) * kColFresh - 1;      // of element 0
    const bool left = col < 0;
    const int last = a.w - col;                            // elements from here on are padding on the right
    int row = (hh ? seg1 : seg0) * a.seg_rows * STRIDE - 1;
    const bool ragged = __builtin_amdgcn_ballot_w64(last < 15) != 0;

    // ---- the lane that stores: 56 lanes, a channel's columns of both units side by side
    constexpr int kRun = 2 * kOut, kPer = 56 / kRun;       // floats of a channel; channels per store
    const int sch = lane / kRun, sidx = lane - sch * kRun;
    const bool shalf = sidx >= kOut;
    const int scol = (shalf ? cu1 : cu0) * kOut + (shalf ? sidx - kOut : sidx);
    int srow = (shalf ? seg1 : seg0) * a.seg_rows;
    const int oplane = a.oh * a.ow;
    const bool stores = lane < 56 && scol < a.ow && (!shalf || second);
    uint32_t soff = (uint32_t)(sch * oplane + srow * a.ow + scol) * 4u;
    const auto ybuf = __builtin_amdgcn_make_buffer_rsrc((void*)(y + ((size_t)n * a.cmid + c0) * oplane), 0,
                                                        kColCB * oplane * 4, kBufferFlags);
    // ---- POOL: which results of this lane's channel and unit exist
    const int pcols = hh && !second ? 0 : a.ow - (hh ? cu1 : cu0) * kOut;
    const bool pragged = POOL && __builtin_amdgcn_ballot_w64(pcols < kOut) != 0;
    int prow = (hh ? seg1 : seg0) * a.seg_rows;
    double psum = 0.0;
    float* const ex_w = &exchange[wave][j * kColPitch + hh * kOut];
    const float* const ex_r = &exchange[wave][sch * kColPitch + sidx];

    // the next image row of both units: its sixteen activated columns, zero outside the image
    auto expand = [&](float (&e)[16]) {
        floatx16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll
        for (int s = 0; s < CHUNKS * 8; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(px[s], wr[s], acc, 0, 0, 0);
        load_row();
#pragma unroll
        for (int i = 0; i < 16; ++i) e[i] = acc[i] + bias1;
        col_activate<SWISH>(e, a.act1);
        const bool outside = row < 0 || row >= a.h;
        if (ragged || __builtin_amdgcn_ballot_w64(outside) != 0) {
            const int end = outside ? 0 : last;
#pragma unroll
            for (int i = 0; i < 15; ++i) e[i] = i < end ? e[i] : 0.f;
            e[15] = outside ? 0.f : e[15];
        }
        e[0] = left ? 0.f : e[0];                          // a whole last unit has one column of padding, too
        e[15] = last < 16 ? 0.f : e[15];
        ++row;
    };
    auto stencil_row = [&](float (&s)[kOut], const float (&e)[16], int ky) {
#pragma unroll
        for (int o = 0; o < kOut; ++o)
#pragma unroll
            for (int kx = 0; kx < 3; ++kx) s[o] += taps[ky * 3 + kx] * e[o * STRIDE + kx];
    };
    auto store = [&](float (&s)[kOut]) {
        col_activate<SWISH>(s, a.act2);
#pragma unroll
        for (int o = 0; o < kOut; ++o) ex_w[o] = s[o];
        if constexpr (POOL) {
            float r = 0.f;
            if (pragged) {
#pragma unroll
                for (int o = 0; o < kOut; ++o) r += o < pcols ? s[o] : 0.f;
            } else {
#pragma unroll
                for (int o = 0; o < kOut; ++o) r += s[o];
            }
            psum += (double)(prow < a.oh ? r : 0.f);
            ++prow;
        }
        // LDS operations of one wavefront take effect in order: only the compiler has to keep them so
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (stores && srow < a.oh) {
#pragma unroll
            for (int k = 0; k < kColCB / kPer; ++k)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, ex_r[k * kPer * kColPitch]), ybuf, soff,
                                                      k * kPer * oplane * 4, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        ++srow;
        soff += (uint32_t)a.ow * 4u;
    };
    auto start = [&](float (&s)[kOut]) {
#pragma unroll
        for (int o = 0; o < kOut; ++o) s[o] = bias2;
    };

    float e[16];
    if constexpr (STRIDE == 2) {
        float s0[kOut];
        expand(e);
        start(s0);
        stencil_row(s0, e, 0);
        for (int r = 0; r < a.seg_rows; ++r) {
            expand(e);
            stencil_row(s0, e, 1);
            expand(e);
            stencil_row(s0, e, 2);
            store(s0);
            start(s0);
            stencil_row(s0, e, 0);
        }
    } else {
        float s0[kOut], s1[kOut];                          // sums that have seen two rows, one row
        expand(e);
        start(s0);
        stencil_row(s0, e, 0);
        expand(e);
        stencil_row(s0, e, 1);
        start(s1);
        stencil_row(s1, e, 0);
        for (int r = 0; r < a.seg_rows; ++r) {
            expand(e);
            stencil_row(s0, e, 2);
            store(s0);
            stencil_row(s1, e, 1);
#pragma unroll
            for (int o = 0; o < kOut; ++o) s0[o] = s1[o];
            start(s1);
            stencil_row(s1, e, 0);
        }
    }
    if constexpr (POOL) {
        psum += __shfl_xor(psum, 32);   // both units
        if (lane < 32) a.sums[((size_t)n * a.pairs + pair) * a.cmid + c0 + j] = (float)psum;
    }
}

// The mean of an image's channel from its wavefronts' sums: sixteen channels of one image per workgroup, sixteen lanes each, a
// lane's first eight loads in flight together (2 - 3 us, a launch that waits for memory once).
__global__ __launch_bounds__(256) void pool_columns_kernel(const float* __restrict__ sums, float* __restrict__ pooled, int cmid,
                                                           int pairs, double pixels) {
    __shared__ double share[16][17];
    const int c = threadIdx.x & 15, slot = threadIdx.x >> 4;
    const uint32_t per = (uint32_t)cmid / 16u;
    const uint32_t n = blockIdx.x / per, c0 = (blockIdx.x - n * per) * 16u;
    const float* p = sums + (size_t)n * pairs * cmid + c0 + c;
    double s = 0.0;
    for (int q0 = slot; q0 < pairs; q0 += 128) {
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = p[(size_t)min(q0 + 16 * i, pairs - 1) * cmid];
#pragma unroll
        for (int i = 0; i < 8; ++i) s += (double)(q0 + 16 * i < pairs ? v[i] : 0.f);
    }
    share[slot][c] = s;
    __syncthreads();
    if (slot == 0) {
        s = 0.0;
#pragma unroll
        for (int q = 0; q < 16; ++q) s += share[q][c];
        pooled[(size_t)n * cmid + c0 + c] = (float)(s / pixels);
    }
}

template <int CHUNKS, bool POOL>
int launch_columns(const ColArgs& a, int stride, const float* x, const float* we, const float* be, const float* wd,
                   const float* bd, float* y, hipStream_t st) {
    const bool swish = a.act1 == DMLHIP_ACT_SWISH && a.act2 == DMLHIP_ACT_SWISH;
    const auto kern = stride == 1 ? (swish ? expand_depthwise_columns_kernel<CHUNKS, 1, true, POOL> : expand_depthwise_columns_kernel<CHUNKS, 1, false, POOL>)
                                  : (swish ? expand_depthwise_columns_kernel<CHUNKS, 2, true, POOL> : expand_depthwise_columns_kernel<CHUNKS, 2, false, POOL>);
    note_conv_form(16);
    hipLaunchKernelGGL(kern, a.blocks, kColWaves * 64, 0, st, x, we, be, wd, bd, y, a);
    return launch_status("conv2d_expand_depthwise");
}

int column_compute_units() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 256;
    return cus > 0 ? cus : 256;
}

size_t column_sums_bytes(int64_t n, int64_t cmid, int64_t pairs) { return (size_t)(n * pairs * cmid) * sizeof(float); }

// How the kernel above runs a problem, with no more than `most` bytes of sums; false: the kernels with the expanded rows in LDS
// have to run
bool plan_columns(const dmlhip_conv2d_desc& pw, int stride, int act2, size_t most, ColArgs& a) {
    const int64_t n = pw.n, cin = pw.c, cmid = pw.m, h = pw.h, w = pw.w;
    const int act1 = pw.act;
    if (cin > kColMaxCin) return false;
    const bool swish = act1 == DMLHIP_ACT_SWISH || act2 == DMLHIP_ACT_SWISH, relu = act1 == DMLHIP_ACT_RELU || act2 == DMLHIP_ACT_RELU;
    if (act1 == DMLHIP_ACT_SIGMOID || act2 == DMLHIP_ACT_SIGMOID || (swish && relu)) return false;   // as the other kernels
    // where not one row fits the other kernels' LDS the call stays refused
    if (expand_depthwise_pinned() || dmlhip_conv2d_expand_depthwise_lds_bytes(w, cin, stride) == 0) return false;
    a.sums = nullptr;
    a.cmid = (int)cmid; a.h = (int)h; a.w = (int)w; a.act1 = act1; a.act2 = act2;
    a.oh = (int)((h - 1) / stride + 1);
    a.ow = (int)((w - 1) / stride + 1);
    // an image's input and a channel block's output are addressed with 32-bit byte offsets
    if (cin * h * w >= (1LL << 29) || (int64_t)kColCB * a.oh * a.ow >= (1LL << 29)) return false;
    const int out = kColFresh / stride;
    a.cunits = (a.ow + out - 1) / out;
    a.cblocks = (uint32_t)(cmid / kColCB);
    // Where the other kernels are the faster ones, us there and here. Columns past the image are computed for nothing:
    // [96,32,17,17] -> 192 30.0 and 31.2, [24,16,43,43] -> 96 18.0 and 19.4. A wavefront's loads of weights and its chain of
    // rows take 7 - 9 us however little there is to do, and images of up to 42 columns have few units: [4,32,28,28] -> 192,
    // stride 2, 6.1 and 8.5 (24 images 14.6 and 9.7), [24,32,14,14] -> 192 6.7 and 8.8. More channels cost registers and matrix
    // instructions: [4,48,30,30] -> 96 7.4 and 10.9, [24,48,28,28] -> 288, stride 2, 17.4 and 18.6 ([24,48,56,56] 59.6 and 41.2),
    // [96,80,14,14] -> 480 50 and 56, [96,64,28,28] -> 384 102 and 110.
    const int64_t rows_of_units = n * a.cblocks * h * a.cunits;
    if (5 * w < 4LL * kColFresh * a.cunits || (w <= 42 && (cin > 32 || rows_of_units < 4000)) || (cin > 32 && rows_of_units < 8000))
        return false;
    // Output rows of a unit: each unit expands its first rows (3 - stride of them) once more and starts without loads in
    // flight, so few; but a SIMD has the throughput of about three wavefronts. Cost in image rows of the busiest SIMD.
    const long long simds = 4LL * column_compute_units();
    long long best = -1;
    for (int segs = 1; segs <= a.oh; segs *= 2) {
        const int rows = (a.oh + segs - 1) / segs;
        const long long units = (long long)a.cunits * ((a.oh + rows - 1) / rows);
        const long long waves = (long long)n * a.cblocks * ((units + 1) / 2);
        if (waves > 0x3fffffffLL || units > 0x3fffffffLL || column_sums_bytes(n, cmid, (units + 1) / 2) > most) break;
        const long long cost = std::max(3LL, (waves + simds - 1) / simds) * ((rows - 1) * stride + 3 + 1);
        if (best < 0 || cost < best) {
            best = cost;
            a.seg_rows = rows;
            a.units = (int)units;
            a.pairs = (uint32_t)((units + 1) / 2);
            a.total = (uint32_t)waves;
        }
    }
    if (best < 0) return false;
    a.blocks = (a.total + kColWaves - 1) / kColWaves;
    return true;
}

template <bool POOL>
int launch_columns(const ColArgs& a, int64_t cin, int stride, const float* x, const float* we, const float* be, const float* wd,
                   const float* bd, float* y, hipStream_t st) {
    switch (cin / 16) {
        case 1: return launch_columns<1, POOL>(a, stride, x, we, be, wd, bd, y, st);
        case 2: return launch_columns<2, POOL>(a, stride, x, we, be, wd, bd, y, st);
        default: return launch_columns<3, POOL>(a, stride, x, we, be, wd, bd, y, st);
    }
}

int check_expand_depthwise(const dmlhip_conv2d_desc* pw, const dmlhip_conv2d_desc* dw) {
    DML_REQUIRE(pw && dw, DMLHIP_ERR_NULL, "conv2d_expand_depthwise: NULL descriptor");
    DML_REQUIRE(pw->n >= 0 && pw->c > 0 && pw->h > 0 && pw->w > 0 && pw->m > 0, DMLHIP_ERR_SHAPE,
                "conv2d_expand_depthwise: extents must be positive");
    DML_REQUIRE(valid_act(pw->act) && valid_act(dw->act) && pw->act != DMLHIP_ACT_GELU && dw->act != DMLHIP_ACT_GELU,
                DMLHIP_ERR_ENUM, "conv2d_expand_depthwise: unsupported activation");
    const bool pointwise = pw->kh == 1 && pw->kw == 1 && pw->stride_h == 1 && pw->stride_w == 1 && pw->pad_h == 0 &&
                           pw->pad_w == 0 && pw->group == 1;
    const bool depthwise = dw->kh == 3 && dw->kw == 3 && dw->pad_h == 1 && dw->pad_w == 1 && dw->dil_h == 1 &&
                           dw->dil_w == 1 && dw->stride_h == dw->stride_w && (dw->stride_h == 1 || dw->stride_h == 2) &&
                           dw->group == dw->c && dw->m == dw->c;
    DML_REQUIRE(pointwise && depthwise, DMLHIP_ERR_UNSUPPORTED,
                "conv2d_expand_depthwise: needs a 1x1 / stride 1 / unpadded convolution followed by a 3x3 depthwise "
                "convolution with padding 1 and stride 1 or 2");
    DML_REQUIRE(dw->n == pw->n && dw->c == pw->m && dw->h == pw->h && dw->w == pw->w, DMLHIP_ERR_SHAPE,
                "conv2d_expand_depthwise: the depthwise input must be the pointwise output");
    DML_REQUIRE(pw->c % 16 == 0 && pw->m % kColCB == 0, DMLHIP_ERR_UNSUPPORTED,
                "conv2d_expand_depthwise: needs input channels %% 16 == 0 and expanded channels %% 32 == 0");
    DML_REQUIRE(pw->h * pw->w < (1LL << 30) && pw->w <= 4096 && pw->c * pw->h * pw->w < (1LL << 31), DMLHIP_ERR_UNSUPPORTED,
                "conv2d_expand_depthwise: image too large");
    return 0;
}

}  // namespace
}  // namespace dml

using namespace dml;

extern "C" {

int dmlhip_conv2d_expand_depthwise_f32(const dmlhip_conv2d_desc* pw, const dmlhip_conv2d_desc* dw, const void* x,
                                       const void* w_pw, const void* b_pw, const void* w_dw, const void* b_dw, void* y,
                                       void* stream) {
    if (int e = check_expand_depthwise(pw, dw)) return e;
    if (pw->n == 0) return 0;
    DML_REQUIRE(x && w_pw && w_dw && y, DMLHIP_ERR_NULL, "conv2d_expand_depthwise: NULL tensor pointer");
    ColArgs a;
    if (plan_columns(*pw, (int)dw->stride_h, dw->act, SIZE_MAX, a))
        return launch_columns<false>(a, pw->c, (int)dw->stride_h, (const float*)x, (const float*)w_pw, (const float*)b_pw,
                                     (const float*)w_dw, (const float*)b_dw, (float*)y, (hipStream_t)stream);
    return launch_expand_depthwise_lds(pw, dw, x, w_pw, b_pw, w_dw, b_dw, y, (hipStream_t)stream);
}

size_t dmlhip_conv2d_expand_depthwise_pool_workspace_bytes(const dmlhip_conv2d_desc* pw, const dmlhip_conv2d_desc* dw) {
    ColArgs a;
    if (check_expand_depthwise(pw, dw) || pw->n == 0 || !plan_columns(*pw, (int)dw->stride_h, dw->act, SIZE_MAX, a)) return 0;
    return column_sums_bytes(pw->n, pw->m, a.pairs);
}

int dmlhip_conv2d_expand_depthwise_pool_f32(const dmlhip_conv2d_desc* pw, const dmlhip_conv2d_desc* dw, const void* x,
                                            const void* w_pw, const void* b_pw, const void* w_dw, const void* b_dw, void* y,
                                            void* pooled, void* workspace, size_t workspace_bytes, void* stream) {
    if (int e = check_expand_depthwise(pw, dw)) return e;
    if (pw->n == 0) return 0;
    DML_REQUIRE(x && w_pw && w_dw && y && pooled, DMLHIP_ERR_NULL, "conv2d_expand_depthwise_pool: NULL tensor pointer");
    const int stride = (int)dw->stride_h;
    ColArgs a;
    if (!plan_columns(*pw, stride, dw->act, workspace ? workspace_bytes : 0, a)) {
        if (int e = dmlhip_conv2d_expand_depthwise_f32(pw, dw, x, w_pw, b_pw, w_dw, b_dw, y, stream)) return e;
        const int64_t pixels = ((pw->h - 1) / stride + 1) * ((pw->w - 1) / stride + 1);
        return dmlhip_reduce_f32(DMLHIP_RMEAN, y, pooled, DMLHIP_F32, pw->n * pw->m, pixels, 1, nullptr, 0, stream);
    }
    a.sums = (float*)workspace;
    if (int e = launch_columns<true>(a, pw->c, stride, (const float*)x, (const float*)w_pw, (const float*)b_pw,
                                     (const float*)w_dw, (const float*)b_dw, (float*)y, (hipStream_t)stream)) return e;
    hipLaunchKernelGGL(pool_columns_kernel, (unsigned)(pw->n * (a.cmid / 16)), 256, 0, (hipStream_t)stream, a.sums, (float*)pooled,
                       a.cmid, (int)a.pairs, (double)a.oh * a.ow);
    return launch_status("conv2d_expand_depthwise_pool");
}

}  // extern "C"
