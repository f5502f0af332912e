// Runs a list of entry point calls: what a program launches per step, for one call from the host language instead of one for each
// kernel. 27 launches of 1.5 - 9 us that a Python program issues one by one take it 93 us.
#include "common.h"

#include <string.h>

#include <type_traits>
#include <utility>

namespace {

// An argument as its parameter's type
template <typename T>
T from_word(uint64_t v) {
    if constexpr (std::is_pointer_v<T>) {
        return reinterpret_cast<T>(static_cast<uintptr_t>(v));
    } else if constexpr (std::is_same_v<T, float>) {
        const uint32_t bits = static_cast<uint32_t>(v);
        float f;
        memcpy(&f, &bits, sizeof f);
        return f;
    } else {
        static_assert(std::is_integral_v<T>, "parameters are pointers, integers and floats");
        return static_cast<T>(v);
    }
}

template <typename... A, size_t... I>
int invoke(int (*fn)(A...), const uint64_t* v, std::index_sequence<I...>) {
    return fn(from_word<A>(v[I])...);
}

template <typename... A>
constexpr int arity(int (*)(A...)) {
    return (int)sizeof...(A);
}

template <auto F, int N>
int thunk(const uint64_t* v) {
    return invoke(F, v, std::make_index_sequence<N>{});
}

struct Entry {
    const char* name;
    int argc;
    int (*run)(const uint64_t*);
};

// every entry point that launches kernels: int results, the stream last
#define DML_ENTRY_POINTS(X) \
    X(dmlhip_softmax_f16) \
    X(dmlhip_softmax_f32) \
    X(dmlhip_softmax_backward_f16) \
    X(dmlhip_softmax_backward_f32) \
    X(dmlhip_log_softmax_f16) \
    X(dmlhip_log_softmax_f32) \
    X(dmlhip_log_softmax_backward_f16) \
    X(dmlhip_log_softmax_backward_f32) \
    X(dmlhip_layernorm_f16) \
    X(dmlhip_layernorm_f32) \
    X(dmlhip_layernorm_backward_f16) \
    X(dmlhip_layernorm_backward_grads_f16) \
    X(dmlhip_layernorm_backward_f32) \
    X(dmlhip_layernorm_backward_noalloc_f16) \
    X(dmlhip_batchnorm_inference_f16) \
    X(dmlhip_batchnorm_inference_f32) \
    X(dmlhip_batchnorm_training_f16) \
    X(dmlhip_batchnorm_training_f32) \
    X(dmlhip_batchnorm_backward_f16) \
    X(dmlhip_batchnorm_backward_f32) \
    X(dmlhip_batchnorm_inference_act_f16) \
    X(dmlhip_batchnorm_inference_act_f32) \
    X(dmlhip_batchnorm_training_act_f16) \
    X(dmlhip_batchnorm_training_act_f32) \
    X(dmlhip_batchnorm_backward_act_f16) \
    X(dmlhip_batchnorm_backward_act_f32) \
    X(dmlhip_binary_f16) \
    X(dmlhip_binary_f32) \
    X(dmlhip_unary_f16) \
    X(dmlhip_unary_f32) \
    X(dmlhip_unary_backward_f16) \
    X(dmlhip_unary_backward_f32) \
    X(dmlhip_sum_f16) \
    X(dmlhip_sum_f32) \
    X(dmlhip_bias_gelu_f16) \
    X(dmlhip_bias_gelu_f32) \
    X(dmlhip_cast) \
    X(dmlhip_reduce_f16) \
    X(dmlhip_reduce_f32) \
    X(dmlhip_row_affine_f16) \
    X(dmlhip_row_affine_f32) \
    X(dmlhip_row_dot_f16) \
    X(dmlhip_row_dot_f32) \
    X(dmlhip_transpose_f16) \
    X(dmlhip_transpose_f32) \
    X(dmlhip_maxpool2d_f16) \
    X(dmlhip_maxpool2d_f32) \
    X(dmlhip_maxpool2d_backward_f16) \
    X(dmlhip_maxpool2d_backward_f32) \
    X(dmlhip_pad_constant_f16) \
    X(dmlhip_pad_constant_f32) \
    X(dmlhip_gemm_f16) \
    X(dmlhip_gemm_f16_ws) \
    X(dmlhip_gemm_f16_grouped) \
    X(dmlhip_gemm_f16_grouped_asum) \
    X(dmlhip_gemm_f16_ksum) \
    X(dmlhip_gemm_f32) \
    X(dmlhip_conv2d_f32) \
    X(dmlhip_conv2d_f16) \
    X(dmlhip_conv2d_gated_f32) \
    X(dmlhip_conv2d_expand_depthwise_f32) \
    X(dmlhip_conv2d_expand_depthwise_pool_f32) \
    X(dmlhip_conv2d_backward_data_f32) \
    X(dmlhip_conv2d_backward_weight_f32) \
    X(dmlhip_reduce_sum_multi_f16) \
    X(dmlhip_reduce_sum_multi_f32) \
    X(dmlhip_attention_f16) \
    X(dmlhip_attention_backward_f16) \
    X(dmlhip_attention_masked_f16) \
    X(dmlhip_attention_masked_backward_f16)

constexpr int kMostArguments = 32, kMostTable = 16;
#define DML_ENTRY(F) {#F, arity(&F), &thunk<&F, arity(&F)>},
const Entry kEntries[] = {DML_ENTRY_POINTS(DML_ENTRY)};
#undef DML_ENTRY
#define DML_FITS(F) static_assert(arity(&F) <= kMostArguments, #F);
DML_ENTRY_POINTS(DML_FITS)
#undef DML_FITS
constexpr int kCount = (int)(sizeof(kEntries) / sizeof(kEntries[0]));

}  // namespace

extern "C" {

int dmlhip_call_symbol(const char* name) {
    for (int i = 0; name && i < kCount; ++i)
        if (!strcmp(kEntries[i].name, name)) return i;
    return -1;
}

int dmlhip_run_calls(const dmlhip_call* calls, int count, const uint64_t* pointers, void* stream, int* failed) {
    if (failed) *failed = -1;
    DML_REQUIRE(count >= 0, DMLHIP_ERR_SHAPE, "run_calls: negative count");
    DML_REQUIRE(count == 0 || calls, DMLHIP_ERR_NULL, "run_calls: NULL list");
    for (int i = 0; i < count; ++i) {
        if (failed) *failed = i;
        const dmlhip_call& c = calls[i];
        DML_REQUIRE(c.symbol >= 0 && c.symbol < kCount, DMLHIP_ERR_ENUM, "run_calls: unknown entry point %d", c.symbol);
        DML_REQUIRE(c.args && c.argc == kEntries[c.symbol].argc, DMLHIP_ERR_SHAPE, "run_calls: %s takes %d arguments, got %d",
                    kEntries[c.symbol].name, kEntries[c.symbol].argc, c.argc);
        uint64_t words[kMostArguments], tables[4][kMostTable];
        int used = 0;
        for (int k = 0; k < c.argc; ++k) {
            const dmlhip_call_arg& a = c.args[k];
            switch (a.kind) {
                case DMLHIP_CALL_VALUE: words[k] = a.value; break;
                case DMLHIP_CALL_POINTER:
                    DML_REQUIRE(pointers, DMLHIP_ERR_NULL, "run_calls: NULL pointers");
                    words[k] = pointers[a.index] + a.value;
                    break;
                case DMLHIP_CALL_STREAM: words[k] = reinterpret_cast<uintptr_t>(stream); break;
                case DMLHIP_CALL_TABLE: {
                    DML_REQUIRE(pointers && a.value && used < 4 && a.index <= kMostTable, DMLHIP_ERR_SHAPE, "run_calls: bad pointer table");
                    const dmlhip_call_arg* entries = reinterpret_cast<const dmlhip_call_arg*>(static_cast<uintptr_t>(a.value));
                    for (uint32_t e = 0; e < a.index; ++e) tables[used][e] = pointers[entries[e].index] + entries[e].value;
                    words[k] = reinterpret_cast<uintptr_t>(tables[used++]);
                    break;
                }
                default: DML_REQUIRE(false, DMLHIP_ERR_ENUM, "run_calls: bad argument kind %u", a.kind);
            }
        }
        if (const int e = kEntries[c.symbol].run(words)) return e;
    }
    if (failed) *failed = -1;
    return 0;
}

}  // extern "C"
