// Raw quant bytes to fp16: the arithmetic that the kernels which decode weights have in common
// (jl_gemm_skinny_kernels.h and jl_gemm_reg.hip; of it jl_gemm.hip and jl_gemm_dense.hip take bytes_to_h2).
#pragma once

#include "jl_device.h"
#include "jl_internal.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// ---- raw block bytes -> fp16 fragments of eight consecutive columns ----
//
// A byte b in 0..255 under the exponent byte 0x64 is the fp16 number 1024 + b, exactly; a packed
// subtract recentres it and a packed multiply applies the block scale.  Each product is exact
// before its one rounding, so a decoded weight is the host's float decode rounded once to fp16.

// `sel` picks two bytes of v (selector values 4..7) and pairs each with 0x64 (selector 0).
__device__ __forceinline__ h2 bytes_to_h2(uint32_t v, uint32_t sel) {
    return __builtin_bit_cast(h2, __builtin_amdgcn_perm(v, 0x64646464u, sel));
}

// eight bytes (two dwords, already in 0..255 offset form) -> (byte - bias) * d
__device__ __forceinline__ half8 frag_scaled(uint32_t q0, uint32_t q1, h2 bias, h2 d) {
    h2 a = (bytes_to_h2(q0, 0x00050004u) - bias) * d;
    h2 b = (bytes_to_h2(q0, 0x00070006u) - bias) * d;
    h2 c = (bytes_to_h2(q1, 0x00050004u) - bias) * d;
    h2 e = (bytes_to_h2(q1, 0x00070006u) - bias) * d;
    return half8{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
}

// eight nibbles (two dwords of bytes 0..15) -> the exact integers q * sc: (1024 + q) * sc - 1024 sc
// in one fused step, so the only rounding would be that of the (exact) result
__device__ __forceinline__ half8 frag_times(uint32_t q0, uint32_t q1, h2 sc, h2 off) {
    h2 a = __builtin_elementwise_fma(bytes_to_h2(q0, 0x00050004u), sc, off);
    h2 b = __builtin_elementwise_fma(bytes_to_h2(q0, 0x00070006u), sc, off);
    h2 c = __builtin_elementwise_fma(bytes_to_h2(q1, 0x00050004u), sc, off);
    h2 e = __builtin_elementwise_fma(bytes_to_h2(q1, 0x00070006u), sc, off);
    return half8{a[0], a[1], b[0], b[1], c[0], c[1], e[0], e[1]};
}

// Bytes of 256 columns of a row (four slices): every type's blocks tile 256 columns exactly.
constexpr int quad_bytes(int type) {
    return type == JL_Q8_0 ? 272 : type == JL_Q4_0 ? 144 : type == JL_Q4_K ? 144 : type == JL_Q6_K ? 210
           : type == JL_Q5_K ? 176 : type == JL_Q4_1 ? 160 : type == JL_Q5_0 ? 176 : type == JL_IQ4_XS ? 136 : 0;
}
// Types whose 256-column block has one scale for everything a wave's MFMAs add up: the fragments
// hold small integers (sub-block scale x quant) and the block's d multiplies the MFMA result.
template <int TYPE> constexpr bool kPostScale = TYPE == JL_Q4_K || TYPE == JL_Q5_K || TYPE == JL_Q6_K || TYPE == JL_IQ4_XS;
// Types with an additive term per 32 columns (a minimum), folded in by one more MFMA against the
// activations' sums over those 32 columns.
template <int TYPE> constexpr bool kHasMins = TYPE == JL_Q4_K || TYPE == JL_Q5_K || TYPE == JL_Q4_1;

// a signed byte of `v` as a pair of equal fp16 values
__device__ __forceinline__ h2 sbyte_h2(uint32_t v, int byte) {
    const _Float16 f = (_Float16)(float)(int)(int8_t)(v >> (8 * byte));
    return h2{f, f};
}

}  // namespace
