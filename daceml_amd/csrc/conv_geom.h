// Geometry of a 2-D convolution after validation (all extents fit an int): shared by the convolution sources.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dml {

struct ConvGeom {
    int n, c, h, w, m, kh, kw, sh, sw, ph, pw, dh, dw, group, oh, ow, cg, mg, act;
};

// conv_implicit.hip: does the general implicit-GEMM kernel take the convolution / its data gradient
bool conv_implicit_applicable(const ConvGeom& g);
bool conv_implicit_bwd_data_applicable(const ConvGeom& g);

// conv_dense3.hip: 3 x 3, group 1, with enough work. *applies = false: nothing launched, another kernel has to run
int launch_conv_dense3_f32(const ConvGeom& g, const float* x, const float* w, const float* bias, float* y, hipStream_t st,
                           bool* applies);
int launch_conv_dense3_bwd_data_f32(const ConvGeom& g, const float* dy, const float* w, float* dx, hipStream_t st, bool* applies);
// its estimate, < 0: does not apply; *chains: sums that it cuts the input channels into
double conv_dense3_us(const ConvGeom& g, int ids_h, int ids_w, bool flip, const void* x, const void* w, int* chains);
void note_conv_form(int form);             // diagnostic, this thread: what dmlhip_debug_last_conv_form returns
void conv_dense3_force_tile(int tile);     // diagnostic, this thread: -1 = chosen per problem
// conv_dense3_split.hip: the same problems on the bf16 matrix instructions, where that is faster
int launch_conv_dense3_split_f32(const ConvGeom& g, const float* x, const float* w, const float* bias, float* y, hipStream_t st,
                                 bool* applies);
int launch_conv_dense3_split_bwd_data_f32(const ConvGeom& g, const float* dy, const float* w, float* dx, hipStream_t st, bool* applies);
// conv_dense3_weight.hip: per-range results (m * c * 9 floats each) its weight gradient writes; 0 = does not apply, or the
// general kernel, where that applies (`general`), is the faster one
int64_t conv_dense3_bwd_weight_partials(const ConvGeom& g, bool general);
// ... on the bf16 matrix instructions (conv_dense3_weight_split.hip) or the fp32 one
int launch_conv_dense3_weight(const ConvGeom& g, const float* x, const float* dy, float* part, hipStream_t st);
int launch_conv_dense3_bwd_weight(const ConvGeom& g, const float* x, const float* dy, float* part, hipStream_t st);

// conv_depthwise.hip: depthwise 3 x 3 / 5 x 5, stride 1, output as large as the input
bool depthwise_same_applicable(const ConvGeom& g);
// ... and are they the faster ones, where the general depthwise kernels take the problem too (data: the data gradient)
bool depthwise_same_faster(const ConvGeom& g, const void* in, const void* out, bool data);
bool depthwise_same_weight_faster(const ConvGeom& g, const void* x, const void* dy);
int launch_depthwise_same(const ConvGeom& g, const float* x, const float* w, const float* bias, float* y, hipStream_t st);
int launch_depthwise_same_bwd_data(const ConvGeom& g, const float* dy, const float* w, float* dx, hipStream_t st);
int launch_depthwise_same_bwd_weight(const ConvGeom& g, const float* x, const float* dy, float* part, hipStream_t st);

// conv_pointwise_few.hip: 1 x 1, few input channels, many output channels; w_transposed: w is [cin][cout]
bool pointwise_few_applicable(int64_t n, int64_t cin, int64_t cout, int64_t hw);
int launch_pointwise_few(const float* x, const float* w, const float* bias, float* y, int n, int cin, int cout, int64_t hw,
                         int act, bool w_transposed, hipStream_t st);

// conv_fused.hip: 1 x 1 expansion + 3 x 3 depthwise with the expanded rows in LDS (validated descriptors); is one of its
// geometries asked for by this thread's diagnostic switches
int launch_expand_depthwise_lds(const dmlhip_conv2d_desc* pw, const dmlhip_conv2d_desc* dw, const void* x, const void* w_pw,
                                const void* b_pw, const void* w_dw, const void* b_dw, void* y, hipStream_t st);
bool expand_depthwise_pinned();

// conv_pointwise_project.hip: 1 x 1, many input channels, few output channels; gate (optional): a factor per image and input channel
bool pointwise_project_applicable(int64_t n, int64_t cin, int64_t cout, int64_t hw, bool w_transposed, bool streams);
bool pointwise_splits_channels(int64_t n, int64_t cin, int64_t cout, int64_t hw);   // few pixels: the tiled GEMM is faster, without a gate
int launch_pointwise_project(const float* x, const float* w, const float* bias, const float* gate, float* y, int n, int cin,
                             int cout, int64_t hw, int act, bool w_transposed, hipStream_t st);

// The data gradient of a dense convolution as a convolution: dX = conv(dY with s - 1 zeros between its elements,
// W with input / output channels exchanged and the taps reversed, stride 1, padding (k - 1) d - p).
inline bool data_gradient_problem(const ConvGeom& f, ConvGeom* b) {
    const int ph = (f.kh - 1) * f.dh - f.ph, pw = (f.kw - 1) * f.dw - f.pw;
    if (f.group != 1 || ph < 0 || pw < 0) return false;
    *b = f;
    b->c = f.m; b->m = f.c;            // channels exchanged
    b->h = f.oh; b->w = f.ow;          // the input is dY ...
    b->oh = f.h; b->ow = f.w;          // ... the output dX
    b->sh = b->sw = 1;
    b->ph = ph; b->pw = pw;
    b->cg = b->c; b->mg = b->m;
    b->act = 0;
    return true;
}

}  // namespace dml
