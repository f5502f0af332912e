// BatchNormalization over NCHW tensors: inference, training forward (batch statistics + running-statistics update)
// and backward. HBM-bound: training reads X twice and writes Y once, backward reads dY and X twice and writes dX.
// A Relu or Swish that follows the normalisation can run inside the same kernels (template parameter ACT): the
// forward applies it before the store, the backward recomputes the normalised value from X and multiplies the incoming
// gradient by the activation's derivative, so neither pass touches the tensor more often than without it.
//
// A channel's data are N segments of HW contiguous elements. Workgroup (c, s) of a grid C x S owns a part of channel c, so
// the launch fills the chip also when C is small. The 16-byte vectors of a channel are counted through all its segments and
// cut into S equal spans, S x C no more than the workgroups that are resident at once; a thread has four vectors of each
// operand on its way, the first ones before the statistics are combined. Where HW is no multiple of a vector, a segment's
// last vector overlaps the one before and its leading elements are left out.
// Measured, us: statistics, apply with Swish, backward sums, backward apply - before (chunks of 4096 elements per segment, one
// load in flight, 4-byte loads where HW is no multiple of 8) and now: 32 x 144 x 56 x 56 fp32 12.5 / 20.1 / 21.5 / 27.8 and
// 9.8 / 18.1 / 18.3 / 26.9 (57.8 MB a tensor, 4.3 to 6.4 TB/s), 55 x 55 18.1 / 25.0 / 24.4 / 32.3 and 9.9 / 17.9 / 19.0 / 26.5,
// 32 x 480 x 14 x 14 11.9 / 13.0 / 13.3 / 13.0 and 4.1 / 5.9 / 5.3 / 7.4, 32 x 24 x 56 x 56 3.6 / 5.2 / 5.1 / 5.7 and
// 3.7 / 5.0 / 5.2 / 6.0; fp16 32 x 144 x 56 x 56 8.9 / 11.5 / 15.0 / 15.9 and 6.6 / 11.2 / 12.6 / 15.4. Skipping the loads behind the
// end of a span by a branch each, instead of loading a vector again, cost more than the loads (12.3 instead of 10.4).
// Pointers or extents that do not allow this (an fp16 segment that is no multiple of 16 bytes, HW below a vector) go
// element by element: segments cut into chunks of at most kChunk, workgroup (c, s) takes the chunks s, s+S, ...
// Statistics are accumulated in fp32 as sums of (x - K) and (x - K)^2 with K the
// channel's first element (shifted-data variance: no cancellation against a large mean), written as per-workgroup
// partials; the second kernel of each pair starts by combining its channel's partials (S <= kMaxSplit of them).
#include <initializer_list>
#include <type_traits>

#include "common.h"

namespace dml {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 4096;
constexpr int kResident = 2048;   // workgroups of kThreads that 256 compute units hold
constexpr int kMaxSplit = 64;

struct BnGeom {
    int64_t n, c, hw;
    int split;                // S
    // vectors (vecs > 0)
    uint32_t vecs;            // of a channel: n * vps, below 2^31
    uint32_t vps;             // of a segment: ceil(hw / V)
    uint32_t span;            // of a workgroup
    uint32_t magic;           // v / vps = v * magic >> shift for every v below 2^31
    int shift;
    int skip;                 // elements of a segment's last vector that the vector before it has
    // element by element (vecs == 0)
    int64_t chunks_per_seg;   // ceil(hw / kChunk)
    int64_t chunks;           // n * chunks_per_seg
};

// A 16-byte vector that is only as aligned as the tensor: fp32 segments of any length begin at a multiple of 4 bytes, which
// is all that a global access of 16 bytes needs. fp16 takes the vector path where segments are 16-byte aligned.
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
template <typename T> struct Vec { typedef typename VecOf<T>::type type; };
template <> struct Vec<float> { typedef floatx4u type; };

enum { kByElement = 0, kVectors = 1, kRaggedVectors = 2 };   // how a kernel walks its part of a channel

// The vectors v0, v0 + kThreads, ... of channel c: where they are, and their values of one or two tensors.
// Four at a time; two where both tensors are fp16, whose eight values per vector would cost a resident workgroup.
template <typename T, int WALK, bool TWO> struct Batch {
    static constexpr int V = VecOf<T>::n, kDepth = TWO && sizeof(T) == 2 ? 2 : 4;
    typename Vec<T>::type a[kDepth], b[kDepth];
    int64_t idx[kDepth];
    int skip[kDepth];

    __device__ __forceinline__ void fetch(const BnGeom& g, int c, uint32_t v0, uint32_t end, const T* pa, const T* pb) {
#pragma unroll
        for (int u = 0; u < kDepth; ++u) {
            const uint32_t v = min(v0 + u * kThreads, end - 1);   // behind the end: a vector that is there, not used
            const uint32_t n = (uint32_t)(((uint64_t)v * g.magic) >> g.shift);
            const uint32_t i = v - n * g.vps;
            skip[u] = WALK == kRaggedVectors && i == g.vps - 1 ? g.skip : 0;
            idx[u] = ((int64_t)n * g.c + c) * g.hw + ((int64_t)i * V - skip[u]);
        }
#pragma unroll
        for (int u = 0; u < kDepth; ++u) {
            a[u] = *reinterpret_cast<const typename Vec<T>::type*>(pa + idx[u]);
            if constexpr (TWO) b[u] = *reinterpret_cast<const typename Vec<T>::type*>(pb + idx[u]);
        }
    }
};

// Walks the workgroup's part of channel c, s of S: `ready()` once, behind the first loads; then f(value of pa, value of pb)
// -> result for every element, stored to `out` if STORE (a branch on the pointer kept the loops apart: fp16 32 x 24 x 55 x 55 in
// inference 5.1 us, 4.5 without). pb is read if TWO.
template <typename T, int WALK, bool TWO, bool STORE, typename R, typename F>
__device__ __forceinline__ void walk(const BnGeom& g, int c, int s, const T* pa, const T* pb, T* out, R&& ready, F&& f) {
    if constexpr (WALK == kByElement) {
        ready();
        for (int64_t ch = s; ch < g.chunks; ch += g.split) {
            const int64_t n = ch / g.chunks_per_seg;
            const int64_t off = (ch - n * g.chunks_per_seg) * kChunk;
            const int64_t len = min((int64_t)kChunk, g.hw - off);
            const int64_t base = (n * g.c + c) * g.hw + off;
            for (int64_t i = threadIdx.x; i < len; i += kThreads) {
                const float r = f(to_f32(pa[base + i]), TWO ? to_f32(pb[base + i]) : 0.f);
                if constexpr (STORE) out[base + i] = from_f32<T>(r);
            }
        }
    } else {
        constexpr int V = VecOf<T>::n;
        const uint32_t begin = (uint32_t)s * g.span, end = min(begin + g.span, g.vecs);
        uint32_t v0 = begin + threadIdx.x;
        Batch<T, WALK, TWO> q;
        constexpr int kDepth = q.kDepth;
        q.fetch(g, c, v0, end, pa, pb);
        ready();
        while (v0 < end) {
#pragma unroll
            for (int u = 0; u < kDepth; ++u) {
                if (v0 + u * kThreads >= end) break;
                typename Vec<T>::type o;
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    if (WALK == kRaggedVectors && j < q.skip[u]) continue;
                    o[j] = from_f32<T>(f(to_f32((T)q.a[u][j]), TWO ? to_f32((T)q.b[u][j]) : 0.f));
                }
                if constexpr (!STORE) continue;
                if (WALK == kRaggedVectors && q.skip[u] > 0) {
#pragma unroll
                    for (int j = 0; j < V; ++j)
                        if (j >= q.skip[u]) out[q.idx[u] + j] = (T)o[j];
                } else {
                    *reinterpret_cast<typename Vec<T>::type*>(out + q.idx[u]) = o;
                }
            }
            v0 += kDepth * kThreads;
            if (v0 < end) q.fetch(g, c, v0, end, pa, pb);
        }
    }
}

// The activation that may follow the normalisation inside the same kernel (NONE, RELU, SWISH), and its derivative
// with respect to the normalised value z — the backward kernels recompute z from X instead of reading a stored copy.
template <int ACT>
__device__ __forceinline__ float bn_act(float z) {
    if constexpr (ACT == DMLHIP_ACT_SWISH) return z * sigmoid_epilogue_f(z);
    else if constexpr (ACT == DMLHIP_ACT_RELU) return fmaxf(z, 0.f);
    else return z;
}
template <int ACT>
__device__ __forceinline__ float bn_act_grad(float z) {
    if constexpr (ACT == DMLHIP_ACT_SWISH) {
        const float sg = sigmoid_epilogue_f(z);
        return sg * (1.0f + z * (1.0f - sg));
    } else if constexpr (ACT == DMLHIP_ACT_RELU) return z > 0.f ? 1.f : 0.f;
    else return 1.f;
}

// partial[(c * S + s) * 2 + {0, 1}] = sum of (x - K), sum of (x - K)^2 over the workgroup's chunks
template <typename T, int WALK>
__global__ __launch_bounds__(kThreads) void bn_stats_kernel(const T* __restrict__ x, float* __restrict__ partial,
                                                            BnGeom g) {
    __shared__ float scratch[kThreads / kWave];
    const int c = blockIdx.x, s = blockIdx.y;
    const float shift = to_f32(x[(int64_t)c * g.hw]);
    float s1 = 0.f, s2 = 0.f;
    walk<T, WALK, false, false>(g, c, s, x, (const T*)nullptr, (T*)nullptr, [] {}, [&](float v, float) {
        const float d = v - shift;
        s1 += d;
        s2 += d * d;
        return 0.f;
    });
    s1 = block_reduce<OpSum, kThreads / kWave>(s1, scratch);
    s2 = block_reduce<OpSum, kThreads / kWave>(s2, scratch);
    if (threadIdx.x == 0) {
        partial[((int64_t)c * g.split + s) * 2 + 0] = s1;
        partial[((int64_t)c * g.split + s) * 2 + 1] = s2;
    }
}

// Sum of the channel's partial pairs, by the first wavefront; every thread gets the result.
__device__ __forceinline__ void combine_partials(const float* partial, int c, int split, float* lds2, float& a, float& b) {
    if (threadIdx.x < kWave) {
        float p0 = 0.f, p1 = 0.f;
        for (int i = threadIdx.x; i < split; i += kWave) {
            p0 += partial[((int64_t)c * split + i) * 2 + 0];
            p1 += partial[((int64_t)c * split + i) * 2 + 1];
        }
        p0 = wave_reduce<OpSum>(p0);
        p1 = wave_reduce<OpSum>(p1);
        if (threadIdx.x == 0) {
            lds2[0] = p0;
            lds2[1] = p1;
        }
    }
    __syncthreads();
    a = lds2[0];
    b = lds2[1];
}

// TRAINING: statistics from `partial`; workgroup s == 0 also writes the saved and the running statistics.
// otherwise: statistics are the given mean / var.
template <typename T, int WALK, bool TRAINING, int ACT>
__global__ __launch_bounds__(kThreads) void bn_apply_kernel(const T* __restrict__ x, const T* __restrict__ scale,
                                                            const T* __restrict__ bias, const T* __restrict__ in_mean,
                                                            const T* __restrict__ in_var, const float* __restrict__ partial,
                                                            T* __restrict__ y, T* __restrict__ out_mean,
                                                            T* __restrict__ out_var, T* __restrict__ saved_mean,
                                                            T* __restrict__ saved_var, float eps, float momentum,
                                                            BnGeom g) {
    __shared__ float lds2[2];
    const int c = blockIdx.x, s = blockIdx.y;
    float mean, a, b;
    walk<T, WALK, false, true>(g, c, s, x, (const T*)nullptr, y, [&] {
        float var;
        if constexpr (TRAINING) {
            float s1, s2;
            combine_partials(partial, c, g.split, lds2, s1, s2);
            const float cnt = (float)(g.n * g.hw);
            const float shift = to_f32(x[(int64_t)c * g.hw]);
            const float dm = s1 / cnt;
            mean = shift + dm;
            var = fmaxf(s2 / cnt - dm * dm, 0.f);   // biased, as np.add.reduce(...) / N
            if (s == 0 && threadIdx.x == 0) {
                saved_mean[c] = from_f32<T>(mean);
                saved_var[c] = from_f32<T>(var);
                out_mean[c] = from_f32<T>(to_f32(in_mean[c]) * momentum + mean * (1.f - momentum));
                out_var[c] = from_f32<T>(to_f32(in_var[c]) * momentum + var * (1.f - momentum));
            }
        } else {
            mean = to_f32(in_mean[c]);
            var = to_f32(in_var[c]);
        }
        a = to_f32(scale[c]) * (1.0f / sqrtf(var + eps));
        b = to_f32(bias[c]);
    }, [&](float v, float) { return bn_act<ACT>((v - mean) * a + b); });   // centred first: no cancellation for large means
}

// partial pairs: sum of dz, sum of dz * (x - mean), with dz = dy * act'(z) the gradient at the normalised value
template <typename T, int WALK, int ACT>
__global__ __launch_bounds__(kThreads) void bn_bwd_stats_kernel(const T* __restrict__ dy, const T* __restrict__ x,
                                                                const T* __restrict__ scale, const T* __restrict__ bias,
                                                                const T* __restrict__ saved_mean,
                                                                const T* __restrict__ saved_var, float eps,
                                                                float* __restrict__ partial, BnGeom g) {
    __shared__ float scratch[kThreads / kWave];
    const int c = blockIdx.x, s = blockIdx.y;
    const float mean = to_f32(saved_mean[c]);
    float a = 0.f, b = 0.f;
    if constexpr (ACT != DMLHIP_ACT_NONE) {
        a = to_f32(scale[c]) * (1.0f / sqrtf(to_f32(saved_var[c]) + eps));
        b = to_f32(bias[c]);
    }
    float s1 = 0.f, s2 = 0.f;
    walk<T, WALK, true, false>(g, c, s, x, dy, (T*)nullptr, [] {}, [&](float v, float d) {
        const float xc = v - mean;
        const float dz = d * bn_act_grad<ACT>(xc * a + b);
        s1 += dz;
        s2 += dz * xc;
        return 0.f;
    });
    s1 = block_reduce<OpSum, kThreads / kWave>(s1, scratch);
    s2 = block_reduce<OpSum, kThreads / kWave>(s2, scratch);
    if (threadIdx.x == 0) {
        partial[((int64_t)c * g.split + s) * 2 + 0] = s1;
        partial[((int64_t)c * g.split + s) * 2 + 1] = s2;
    }
}

// dx = scale * invstd * (dz - mean(dz) - (x - mean) * invstd^2 * mean(dz * (x - mean)))
template <typename T, int WALK, int ACT>
__global__ __launch_bounds__(kThreads) void bn_bwd_apply_kernel(const T* __restrict__ dy, const T* __restrict__ x,
                                                                const T* __restrict__ scale, const T* __restrict__ bias,
                                                                const T* __restrict__ saved_mean,
                                                                const T* __restrict__ saved_var,
                                                                const float* __restrict__ partial, T* __restrict__ dx,
                                                                float* __restrict__ dscale, float* __restrict__ dbias,
                                                                float eps, BnGeom g) {
    __shared__ float lds2[2];
    const int c = blockIdx.x, s = blockIdx.y;
    float mean, b, k0, k1, k2;
    auto ready = [&] {
        float sum_dy, sum_dyxc;
        combine_partials(partial, c, g.split, lds2, sum_dy, sum_dyxc);
        mean = to_f32(saved_mean[c]);
        const float invstd = 1.0f / sqrtf(to_f32(saved_var[c]) + eps);
        if (s == 0 && threadIdx.x == 0) {
            if (dscale) dscale[c] = sum_dyxc * invstd;
            if (dbias) dbias[c] = sum_dy;
        }
        const float cnt = (float)(g.n * g.hw);
        k0 = to_f32(scale[c]) * invstd;
        k1 = sum_dy / cnt;
        k2 = invstd * invstd * sum_dyxc / cnt;
        b = ACT != DMLHIP_ACT_NONE ? to_f32(bias[c]) : 0.f;
    };
    if (!dx) return ready();
    walk<T, WALK, true, true>(g, c, s, x, dy, dx, ready, [&](float v, float d) {
        const float xc = v - mean;
        return k0 * (d * bn_act_grad<ACT>(xc * k0 + b) - k1 - xc * k2);
    });
}

// *walk: how the kernels go over a channel
template <typename T>
int make_geom(const char* what, int64_t n, int64_t c, int64_t hw, std::initializer_list<const void*> tensors, BnGeom* g,
              int* walk) {
    DML_REQUIRE(n > 0 && c > 0 && hw > 0, DMLHIP_ERR_SHAPE, "%s: extents must be positive, got N=%lld C=%lld HW=%lld", what,
                (long long)n, (long long)c, (long long)hw);
    DML_REQUIRE(c <= 0x7fffffff, DMLHIP_ERR_SHAPE, "%s: %lld channels exceed the grid limit", what, (long long)c);
    g->n = n;
    g->c = c;
    g->hw = hw;
    constexpr int64_t V = VecOf<T>::n;
    const int64_t vps = ceil_div(hw, V);
    bool vectors = hw >= V && n <= 0x7fffffff / vps;
    if (sizeof(T) == 2) {
        vectors = vectors && hw % V == 0;
        for (const void* p : tensors) vectors = vectors && (p == nullptr || aligned16(p));
    }
    if (vectors) {
        g->vecs = (uint32_t)(n * vps);
        g->vps = (uint32_t)vps;
        g->skip = (int)(vps * V - hw);
        int l = 0;
        while ((1ll << l) < vps) ++l;
        g->shift = 31 + l;
        g->magic = (uint32_t)(((1ull << g->shift) + vps - 1) / vps);
        // At most one resident round of workgroups and kMaxSplit per channel; beyond that a thread takes as many vectors, up to
        // a batch of four, as leave about three workgroups per compute unit, and more only in whole batches. Measured for 1 - 12
        // vectors per thread, training + backward + inference with and without Swish, us for 1 / 2 / 3 / 4: fp32 8 x 64 x 56 x 56
        // (1600, 832, 576 workgroups ...) 41.3 / 36.7 / 35.4 / 36.2, 16 x 24 x 56 x 56 (1176, 600, ...) 36.5 / 33.5 / 33.3 / 34.6, 8 x 24 x 56 x 56
        // (600, ...) 30.9 / 30.0 / 30.3 / 31.7, 64 x 64 x 28 x 28 59.7 / 51.0 / 49.6 / 49.9; fp16 32 x 16 x 56 x 56 (784, 400, ...) 33.9 / 31.9 /
        // 32.4 / 34.0, 32 x 32 x 56 x 56 (1568, 800, 544, ...) 43.7 / 40.1 / 39.0 / 41.6, 32 x 96 x 56 x 56 86.0 / 76.4 / 74.2 / 76.0.
        int64_t split = kResident / c;
        split = split < 1 ? 1 : split > kMaxSplit ? kMaxSplit : split;
        int64_t each = ceil_div(ceil_div((int64_t)g->vecs, split), (int64_t)kThreads);
        auto wgs = [&] { return ceil_div((int64_t)g->vecs, each * kThreads) * c; };
        if (each == 1 && wgs() > 640) each = 2;
        if (each == 2 && wgs() > 700) each = 3;
        if (each == 3 && wgs() > 900) each = 4;
        if (each > 4) each = ceil_div(each, (int64_t)4) * 4;
        g->span = (uint32_t)(each * kThreads);
        g->split = (int)ceil_div(g->vecs, g->span);
        *walk = g->skip ? kRaggedVectors : kVectors;
        return 0;
    }
    g->vecs = 0;
    g->chunks_per_seg = ceil_div(hw, kChunk);
    g->chunks = n * g->chunks_per_seg;
    // enough workgroups to fill 256 CUs several times over, never more than there are chunks
    int64_t split = ceil_div(2048, c);
    if (split > g->chunks) split = g->chunks;
    if (split > kMaxSplit) split = kMaxSplit;
    g->split = (int)(split < 1 ? 1 : split);
    *walk = kByElement;
    return 0;
}

size_t bn_workspace(int64_t n, int64_t c, int64_t hw) {
    (void)n;
    (void)hw;
    return c > 0 ? (size_t)c * kMaxSplit * 2 * sizeof(float) : 0;
}

// runs `body(std::integral_constant<int, WALK>)`; ragged vectors are fp32's
template <typename T, typename F>
int with_walk(int walk, F&& body) {
    if constexpr (sizeof(T) == 4)
        if (walk == kRaggedVectors) return body(std::integral_constant<int, kRaggedVectors>{});
    return walk == kVectors ? body(std::integral_constant<int, kVectors>{}) : body(std::integral_constant<int, kByElement>{});
}

// runs `body(std::integral_constant<int, ACT>)` for the activation code, or reports an unsupported one
template <typename F>
int with_activation(const char* what, int act, F&& body) {
    switch (act) {
        case DMLHIP_ACT_NONE: return body(std::integral_constant<int, DMLHIP_ACT_NONE>{});
        case DMLHIP_ACT_RELU: return body(std::integral_constant<int, DMLHIP_ACT_RELU>{});
        case DMLHIP_ACT_SWISH: return body(std::integral_constant<int, DMLHIP_ACT_SWISH>{});
        default:
            set_error("%s: activation %d is not one of NONE, RELU, SWISH", what, act);
            return DMLHIP_ERR_ENUM;
    }
}

template <typename T>
int bn_inference(const void* x, const void* scale, const void* bias, const void* mean, const void* var, void* y,
                 int64_t n, int64_t c, int64_t hw, float eps, int act, void* stream) {
    DML_REQUIRE(x && scale && bias && mean && var && y, DMLHIP_ERR_NULL, "batchnorm_inference: NULL pointer");
    BnGeom g;
    int walk;
    if (int e = make_geom<T>("batchnorm_inference", n, c, hw, {x, y}, &g, &walk)) return e;
    return with_activation("batchnorm_inference", act, [&](auto actc) {
        constexpr int ACT = decltype(actc)::value;
        return with_walk<T>(walk, [&](auto walkc) {
            constexpr int WALK = decltype(walkc)::value;
            hipLaunchKernelGGL((bn_apply_kernel<T, WALK, false, ACT>), dim3((unsigned)c, (unsigned)g.split), kThreads, 0,
                               (hipStream_t)stream, (const T*)x, (const T*)scale, (const T*)bias, (const T*)mean, (const T*)var,
                               (const float*)nullptr, (T*)y, (T*)nullptr, (T*)nullptr, (T*)nullptr, (T*)nullptr, eps, 0.f, g);
            return launch_status("batchnorm_inference");
        });
    });
}

template <typename T>
int bn_training(const void* x, const void* scale, const void* bias, const void* in_mean, const void* in_var, void* y,
                void* out_mean, void* out_var, void* saved_mean, void* saved_var, int64_t n, int64_t c, int64_t hw,
                float eps, float momentum, int act, void* workspace, size_t workspace_bytes, void* stream) {
    DML_REQUIRE(x && scale && bias && in_mean && in_var && y && out_mean && out_var && saved_mean && saved_var,
                DMLHIP_ERR_NULL, "batchnorm_training: NULL pointer");
    BnGeom g;
    int walk;
    if (int e = make_geom<T>("batchnorm_training", n, c, hw, {x, y}, &g, &walk)) return e;
    DML_REQUIRE(workspace && workspace_bytes >= bn_workspace(n, c, hw), DMLHIP_ERR_WORKSPACE,
                "batchnorm_training: workspace of %zu bytes needed, got %zu", bn_workspace(n, c, hw), workspace_bytes);
    const dim3 grid((unsigned)c, (unsigned)g.split);
    if (int e = with_walk<T>(walk, [&](auto walkc) {
            hipLaunchKernelGGL((bn_stats_kernel<T, decltype(walkc)::value>), grid, kThreads, 0, (hipStream_t)stream,
                               (const T*)x, (float*)workspace, g);
            return launch_status("batchnorm_training(statistics)");
        }))
        return e;
    return with_activation("batchnorm_training", act, [&](auto actc) {
        constexpr int ACT = decltype(actc)::value;
        return with_walk<T>(walk, [&](auto walkc) {
            constexpr int WALK = decltype(walkc)::value;
            hipLaunchKernelGGL((bn_apply_kernel<T, WALK, true, ACT>), grid, kThreads, 0, (hipStream_t)stream, (const T*)x,
                               (const T*)scale, (const T*)bias, (const T*)in_mean, (const T*)in_var, (const float*)workspace,
                               (T*)y, (T*)out_mean, (T*)out_var, (T*)saved_mean, (T*)saved_var, eps, momentum, g);
            return launch_status("batchnorm_training");
        });
    });
}

template <typename T>
int bn_backward(const void* dy, const void* x, const void* scale, const void* bias, const void* saved_mean,
                const void* saved_var, void* dx, float* dscale, float* dbias, int64_t n, int64_t c, int64_t hw, float eps,
                int act, void* workspace, size_t workspace_bytes, void* stream) {
    DML_REQUIRE(dy && x && scale && saved_mean && saved_var, DMLHIP_ERR_NULL, "batchnorm_backward: NULL pointer");
    DML_REQUIRE(bias || act == DMLHIP_ACT_NONE, DMLHIP_ERR_NULL,
                "batchnorm_backward: the bias is needed to recompute the activation's input");
    DML_REQUIRE(dx || dscale || dbias, DMLHIP_ERR_NULL, "batchnorm_backward: no gradient requested");
    BnGeom g;
    int walk;
    if (int e = make_geom<T>("batchnorm_backward", n, c, hw, {dy, x, dx}, &g, &walk)) return e;
    DML_REQUIRE(workspace && workspace_bytes >= bn_workspace(n, c, hw), DMLHIP_ERR_WORKSPACE,
                "batchnorm_backward: workspace of %zu bytes needed, got %zu", bn_workspace(n, c, hw), workspace_bytes);
    const dim3 grid((unsigned)c, (unsigned)g.split);
    return with_activation("batchnorm_backward", act, [&](auto actc) {
        constexpr int ACT = decltype(actc)::value;
        return with_walk<T>(walk, [&](auto walkc) {
            constexpr int WALK = decltype(walkc)::value;
            hipLaunchKernelGGL((bn_bwd_stats_kernel<T, WALK, ACT>), grid, kThreads, 0, (hipStream_t)stream, (const T*)dy,
                               (const T*)x, (const T*)scale, (const T*)bias, (const T*)saved_mean, (const T*)saved_var, eps,
                               (float*)workspace, g);
            if (int e = launch_status("batchnorm_backward(sums)")) return e;
            hipLaunchKernelGGL((bn_bwd_apply_kernel<T, WALK, ACT>), grid, kThreads, 0, (hipStream_t)stream, (const T*)dy,
                               (const T*)x, (const T*)scale, (const T*)bias, (const T*)saved_mean, (const T*)saved_var,
                               (const float*)workspace, (T*)dx, dscale, dbias, eps, g);
            return launch_status("batchnorm_backward");
        });
    });
}

}  // namespace
}  // namespace dml

using namespace dml;

extern "C" {

size_t dmlhip_batchnorm_workspace_bytes(int64_t n, int64_t c, int64_t hw) { return bn_workspace(n, c, hw); }

#define DML_BN_ENTRIES(SFX, T)                                                                                         \
    int dmlhip_batchnorm_inference_##SFX(const void* x, const void* scale, const void* bias, const void* mean,         \
                                         const void* var, void* y, int64_t n, int64_t c, int64_t hw, float eps,        \
                                         void* stream) {                                                               \
        return bn_inference<T>(x, scale, bias, mean, var, y, n, c, hw, eps, DMLHIP_ACT_NONE, stream);                  \
    }                                                                                                                  \
    int dmlhip_batchnorm_inference_act_##SFX(const void* x, const void* scale, const void* bias, const void* mean,     \
                                             const void* var, void* y, int64_t n, int64_t c, int64_t hw, float eps,    \
                                             int act, void* stream) {                                                  \
        return bn_inference<T>(x, scale, bias, mean, var, y, n, c, hw, eps, act, stream);                              \
    }                                                                                                                  \
    int dmlhip_batchnorm_training_##SFX(const void* x, const void* scale, const void* bias, const void* in_mean,       \
                                        const void* in_var, void* y, void* out_mean, void* out_var, void* saved_mean,  \
                                        void* saved_var, int64_t n, int64_t c, int64_t hw, float eps, float momentum,  \
                                        void* workspace, size_t workspace_bytes, void* stream) {                       \
        return bn_training<T>(x, scale, bias, in_mean, in_var, y, out_mean, out_var, saved_mean, saved_var, n, c, hw,  \
                              eps, momentum, DMLHIP_ACT_NONE, workspace, workspace_bytes, stream);                     \
    }                                                                                                                  \
    int dmlhip_batchnorm_training_act_##SFX(const void* x, const void* scale, const void* bias, const void* in_mean,   \
                                            const void* in_var, void* y, void* out_mean, void* out_var,                \
                                            void* saved_mean, void* saved_var, int64_t n, int64_t c, int64_t hw,       \
                                            float eps, float momentum, int act, void* workspace,                       \
                                            size_t workspace_bytes, void* stream) {                                    \
        return bn_training<T>(x, scale, bias, in_mean, in_var, y, out_mean, out_var, saved_mean, saved_var, n, c, hw,  \
                              eps, momentum, act, workspace, workspace_bytes, stream);                                 \
    }                                                                                                                  \
    int dmlhip_batchnorm_backward_##SFX(const void* dy, const void* x, const void* scale, const void* saved_mean,      \
                                        const void* saved_var, void* dx, float* dscale, float* dbias, int64_t n,       \
                                        int64_t c, int64_t hw, float eps, void* workspace, size_t workspace_bytes,     \
                                        void* stream) {                                                                \
        return bn_backward<T>(dy, x, scale, nullptr, saved_mean, saved_var, dx, dscale, dbias, n, c, hw, eps,          \
                              DMLHIP_ACT_NONE, workspace, workspace_bytes, stream);                                    \
    }                                                                                                                  \
    int dmlhip_batchnorm_backward_act_##SFX(const void* dy, const void* x, const void* scale, const void* bias,        \
                                            const void* saved_mean, const void* saved_var, void* dx, float* dscale,    \
                                            float* dbias, int64_t n, int64_t c, int64_t hw, float eps, int act,        \
                                            void* workspace, size_t workspace_bytes, void* stream) {                   \
        return bn_backward<T>(dy, x, scale, bias, saved_mean, saved_var, dx, dscale, dbias, n, c, hw, eps, act,        \
                              workspace, workspace_bytes, stream);                                                     \
    }

DML_BN_ENTRIES(f16, _Float16)
DML_BN_ENTRIES(f32, float)
#undef DML_BN_ENTRIES

}  // extern "C"
