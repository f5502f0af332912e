// fp32 values as sums of three bf16 values, for products at fp32 precision on the bf16 matrix instructions.
//
// 2^16 x = h + m + l exactly, each the rounding of what the ones before leave: 24 bits are 8 + 8 + 8, and the last bit of the smallest
// fp32 value (2^-149) is the last one of a bf16 (2^-133) times 2^-16; the matrix instruction takes subnormal values as they are. (Without
// the factor operands below 2^-110 lose their last bits: a product of operands around 2^-120 was 3.5e-5 from the exact one.) Sums are of
// 2^32 times their size. Of the nine products of two such sums six matter: h h, h m, m h, m m, h l, l h (the others are below
// 2^-26 of the product, under the rounding of the sum). The bf16 matrix rate is 16 times the fp32 one, so six products take 0.375
// of the time of the fp32 instruction, and 8 products share a rounding of the fp32 accumulator where that instruction rounds every
// two. That makes 12 roundings for sixteen products, more than it has where operands are zero, unless the five small products have a sum
// of their own (mfma_small): 2, and the small sum's are 2^-8 of their size. Error against fp64, 2-norm over 2-norm, one such pair of sums here
// / one sum on the fp32 instruction: 576 products of N(0, 1) 1.4e-7 / 4.3e-7, one operand behind a ReLU 1.0e-7 / 3.0e-7, uniform on [0, 1)
// 1.3e-7 / 3.6e-7; 9216 products 5.9e-7 / 1.7e-6, 5.1e-7 / 1.2e-6, 5.0e-7 / 1.4e-6. (All six products in one sum: behind a ReLU 3.4e-7 and
// 1.4e-6.)
// Infinities, NaN and values from 2^112 on have no such sum: a result that comes out not finite (or above 2^96) has to be
// computed again from the fp32 values.
#pragma once

#include "common.h"

namespace dml {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

struct Pieces {
    bf16x8 h, m, l;
};

constexpr float kSplitScale = 65536.f, kSplitBack = 1.f / (65536.f * 65536.f);   // of operands; what makes sums their own size again

// Thirteen vector instructions for two values. (What a rounding leaves is also a dot product of a packed pair with (-1, 0) or
// (0, -1), nine instructions in all, but v_dot2c_f32_bf16 does not issue beside the matrix pipe: 16 MFMAs with 64 of them took
// 6.0 us where with 64 subtractions they took 3.8.)
__device__ __forceinline__ floatx2 unpack_bf16(uint32_t v) {
    return {__builtin_bit_cast(float, v << 16), __builtin_bit_cast(float, v & 0xffff0000u)};
}
__device__ __forceinline__ void split_pair(floatx2 v, float scale, uint32_t& h, uint32_t& m, uint32_t& l) {
    v = floatx2{v[0] * scale, v[1] * scale};
    h = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    const floatx2 uh = unpack_bf16(h);
    floatx2 r = {v[0] - uh[0], v[1] - uh[1]};
    m = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
    const floatx2 um = unpack_bf16(m);
    r = floatx2{r[0] - um[0], r[1] - um[1]};
    l = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2));
}
__device__ __forceinline__ Pieces split_eight(const float (&v)[8], float scale = kSplitScale) {
    u32x4 h, m, l;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t ph, pm, pl;
        split_pair(floatx2{v[2 * i], v[2 * i + 1]}, scale, ph, pm, pl);
        h[i] = ph;
        m[i] = pm;
        l[i] = pl;
    }
    return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m), __builtin_bit_cast(bf16x8, l)};
}

// Five of the six products, each at most 2^-8 of the sixth, and the sixth
__device__ __forceinline__ floatx16 mfma_small(const Pieces& a, const Pieces& b, floatx16 low) {
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.l, b.h, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.l, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.m, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.m, b.h, low, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.m, low, 0, 0, 0);
}
__device__ __forceinline__ floatx16 mfma_large(const Pieces& a, const Pieces& b, floatx16 acc) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.h, b.h, acc, 0, 0, 0);
}

}  // namespace dml
