// Device-side helpers shared by the kernels: fp16 widening, Q4_K scale unpacking, wave folds.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#define JL_WAVE 64

// A product rounded to fp32 on its own.  The compiler's default is to contract a * b + c into one
// fma -- across statements, through the *_rn intrinsics (plain operators in this toolchain's
// headers), and even into a mixed-precision fma when the sum is then narrowed to fp16 (with a +0
// addend, which also loses the sign of a zero product).  Java never fuses, so wherever a result
// has to carry the host's bits the product passes through a register the compiler cannot look past.
__device__ __forceinline__ float jl_mul_rn(float a, float b) {
    float r = a * b;
    asm volatile("" : "+v"(r));
    return r;
}

// WIDTH (16 or 4) bytes per lane from `base` + wave_off + lane_off to LDS, lane by lane behind `to`; only lane_off differs
// between lanes.  POLICY: cache policy bits (2: non-temporal).
// A buffer load: one scalar offset per instruction where a global load takes a 64-bit address in two vector registers,
// and counted by the compiler as any other load, where a global load to LDS (an instruction of the flat family) makes it
// answer the first use of another loaded value with a wait for everything.
template <int WIDTH, int POLICY = 0>
__device__ __forceinline__ void jl_load_to_lds(const void *base, void *to, int lane_off, int wave_off) {
    typedef __attribute__((address_space(3))) void lds_void;
    static_assert(WIDTH == 16 || WIDTH == 4, "");
    const auto from = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, -1, 0x00020000);
    if constexpr (WIDTH == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void *)to, 16, lane_off, wave_off, 0, POLICY);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void *)to, 4, lane_off, wave_off, 0, POLICY);
}

// IEEE half bits -> float, exact (subnormals included); the device form of Float.float16ToFloat.
__device__ __forceinline__ float jl_half_bits_to_float(uint32_t bits) {
    return __half2float(__ushort_as_half((unsigned short)(bits & 0xFFFFu)));
}

// The 6-bit scale and minimum of sub-block j of a Q4_K super-block, from its 12 packed bytes held
// as three little-endian dwords (Q4_KFloatTensor.getScaleK4 / getMinK4,
// J/tensor/standard/Q4_KFloatTensor.java:68-85).
__device__ __forceinline__ void jl_q4k_scale_min(uint32_t s0, uint32_t s1, uint32_t s2, int j,
                                                 int &sc, int &mn) {
    // byte b of the 12: b < 4 in s0, b < 8 in s1, else s2
    if (j < 4) {
        sc = (s0 >> (8 * j)) & 63;
        mn = (s1 >> (8 * j)) & 63;
    } else {
        int k = j - 4;
        uint32_t lo = (s2 >> (8 * k)) & 0xFF;  // byte j + 4
        uint32_t a = (s0 >> (8 * k)) & 0xFF;   // byte j - 4
        uint32_t b = (s1 >> (8 * k)) & 0xFF;   // byte j
        sc = (int)((lo & 0xF) | ((a >> 6) << 4));
        mn = (int)((lo >> 4) | ((b >> 6) << 4));
    }
}

// Hands a value back to the compiler as one it knows nothing about.  Used on words of four
// byte-sized quants after their nibble mask: the byte -> float conversions then stay the
// single-instruction v_cvt_f32_ubyteN, where the compiler would otherwise see through the mask and
// extract each 4-bit field on its own (a bit-field extract plus a conversion per weight).
__device__ __forceinline__ uint32_t jl_opaque(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}

// The bits 0..3 of x, one to a byte (bit k of x at bit 0 of byte k).
__device__ __forceinline__ uint32_t jl_spread4(uint32_t x) { return ((x & 0xFu) * 0x00204081u) & 0x01010101u; }

// ggml's kvalues_iq4nl (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113;
// J/tensor/standard/IQ4_XSFloatTensor.java:30-32) of the four nibbles held one to a byte in `idx`,
// as four signed bytes: two byte permutes pick entry idx & 7 of each half of the table, a third
// picks the half by bit 3.
__device__ __forceinline__ uint32_t jl_iq4nl_lookup4(uint32_t idx) {
    const uint32_t low3 = idx & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(0xF6EADDCFu, 0xBFAD9881u, low3);   // entries 0..7
    const uint32_t hi = __builtin_amdgcn_perm(0x71594535u, 0x26190D01u, low3);   // entries 8..15
    return __builtin_amdgcn_perm(hi, lo, 0x03020100u | ((idx & 0x08080808u) >> 1));
}

// Sum over the lanes of each aligned group of `width` lanes (a power of two, at most 64).  Every
// lane of a group ends with the group's total.
template <int WIDTH>
__device__ __forceinline__ float jl_group_sum(float v) {
#pragma unroll
    for (int off = WIDTH / 2; off >= 1; off >>= 1) v += __shfl_xor(v, off, JL_WAVE);
    return v;
}

__device__ __forceinline__ float jl_group_sum_dyn(float v, int width) {
    for (int off = width >> 1; off >= 1; off >>= 1) v += __shfl_xor(v, off, JL_WAVE);
    return v;
}

// SiLU(g) * u with the host's arithmetic: g / (float)(1.0 + exp(-g)) in double, then one float
// divide and one float multiply (CpuOperations.swiGLU, J/inference/op/CpuOperations.java:255-260).
__device__ __forceinline__ float jl_swiglu_value(float g, float u) {
    float denom = (float)(1.0 + exp(-(double)g));
    return jl_mul_rn(__fdiv_rn(g, denom), u);
}

// SiLU(g) * u in single precision: g / (1 + exp(-g)) with expf, a few ulp from the host's double
// form and three orders of magnitude inside the fp16 path's tolerance; the double-precision exp
// costs about 150 instructions per output, which matters at T x hidden outputs per call.
__device__ __forceinline__ float jl_swiglu_single(float g, float u) {
    return g / (1.0f + __expf(-g)) * u;
}
// ... with the reciprocal instruction, up to a unit in the last place from the quotient
__device__ __forceinline__ float jl_swiglu_rcp(float g, float u) { return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u; }

// Four consecutive results of an output row stored as binary16 (round to nearest even): one
// 8-byte store when all four lie inside the row and the address allows it.
__device__ __forceinline__ void jl_store4_f16(_Float16 *dst, const float (&v)[4], int valid) {
    typedef _Float16 jl_half4 __attribute__((ext_vector_type(4)));
    if (valid >= 4 && (((uintptr_t)dst) & 7) == 0) {
        *(jl_half4 *)dst = jl_half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e < valid) dst[e] = (_Float16)v[e];
    }
}

// Maximum over the 64 lanes, in every lane: rotations within the rows of 16, then the halves and quarters
// of the wave swapped (a shuffle through LDS per step took six dependent LDS round trips).
__device__ __forceinline__ float jl_wave_max(float v) {
#define JL_ROR(x, N) __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + N, 0xF, 0xF, false))
    v = fmaxf(v, JL_ROR(v, 8));
    v = fmaxf(v, JL_ROR(v, 4));
    v = fmaxf(v, JL_ROR(v, 2));
    v = fmaxf(v, JL_ROR(v, 1));
#undef JL_ROR
    const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
    const auto f = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(f[0]), __uint_as_float(f[1]));
}

// Activations, fp32 -> fp16 with a power-of-two row scale.  One workgroup of 256 threads per row:
// scale = the power of two that brings the row's largest magnitude into [2^11, 2^12);
// a16 = half(x / scale) (the division is exact).  Rows past `rows` are zero-filled.
// The first HELD x 1024 columns are read once and kept in registers between the two passes (largest
// magnitude, conversion), what a longer row has behind them is read twice.  Every load goes out before
// the first value is used, a pass past the row's end re-reads the thread's first columns: under a condition
// each the loads waited for one another, and without the asm the compiler reads a value again rather
// than keep it.
// MARK (rows of whole 256-column blocks): a row with a block that this one scale does not serve has its scale
// marked by a minus sign.  A wave holds one block in each pass.  Such a block lies more than 2^16 below the
// row's largest magnitude, and values of it lie below fp16's normal range, where they lose bits or vanish:
// with block maxima from 2^-16 on, what values lose there is at most 2^-20 of the largest in their block, a two
// hundredth of what rounding to fp16 takes from that.
template <int HELD, bool MARK>
__device__ __forceinline__ void jl_row_to_f16_held(const float *__restrict__ x, _Float16 *__restrict__ a,
                                                   float *__restrict__ row_scale, int k) {
    typedef _Float16 jl_half4 __attribute__((ext_vector_type(4)));
    typedef float jl_float4 __attribute__((ext_vector_type(4)));
    __shared__ float wave_max[4];
    const int tid = threadIdx.x;
    const int first = tid * 4 < k ? tid * 4 : 0;
    jl_float4 v[HELD];
#pragma unroll
    for (int j = 0; j < HELD; j++) {
        const int i = tid * 4 + j * 1024;
        v[j] = *(const jl_float4 *)(x + (i < k ? i : first));
    }
#pragma unroll
    for (int j = 0; j < HELD; j++) asm volatile("" : "+v"(v[j]));
    auto largest = [](const jl_float4 &w) { return fmaxf(fmaxf(fabsf(w[0]), fabsf(w[1])), fmaxf(fabsf(w[2]), fabsf(w[3]))); };
    float amax = 0.f;
#pragma unroll
    for (int j = 0; j < HELD; j++) amax = fmaxf(amax, largest(v[j]));
    for (int i = tid * 4 + HELD * 1024; i < k; i += 1024) amax = fmaxf(amax, largest(*(const jl_float4 *)(x + i)));
    amax = jl_wave_max(amax);
    if ((tid & 63) == 0) wave_max[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
    // Every row is brought to [2^11, 2^12) at its largest magnitude: huge rows stay finite in
    // fp16, tiny rows keep their bits out of fp16's subnormal range, and the power of two is
    // undone exactly in the epilogue.  (amax = f 2^e with f in [0.5, 1): e = its exponent field - 126,
    // not below -100; a row of zeros, infinities or NaN alone keeps its values)
    float scale = 1.f, inv = 1.f;
    if (amax > 0.f && amax < INFINITY) {
        int e = (int)(__float_as_uint(amax) >> 23) - 126;
        e = e < -100 ? -100 : e;
        scale = __uint_as_float((uint32_t)(e - 12 + 127) << 23);
        inv = __uint_as_float((uint32_t)(12 - e + 127) << 23);
    }
    auto put = [&](int i, const jl_float4 &w) {
        *(jl_half4 *)(a + i) = jl_half4{(_Float16)(w[0] * inv), (_Float16)(w[1] * inv), (_Float16)(w[2] * inv), (_Float16)(w[3] * inv)};
    };
    // (a wave looks at its block's smallest values only where none of the others is large enough)
    bool mark = false;
    auto look = [&](const jl_float4 &w) {
        if (__ballot(largest(w) * inv >= 0x1p-5f) != 0) return;
        bool under = false;
#pragma unroll
        for (int e = 0; e < 4; e++) under = under || (w[e] != 0.f && fabsf(w[e]) * inv < 0x1p-14f);
        mark = mark || __ballot(under) != 0;
    };
#pragma unroll
    for (int j = 0; j < HELD; j++) {
        const int i = tid * 4 + j * 1024;
        if (i < k) {
            put(i, v[j]);
            if constexpr (MARK) look(v[j]);
        }
    }
    for (int i = tid * 4 + HELD * 1024; i < k; i += 1024) {
        const jl_float4 w = *(const jl_float4 *)(x + i);
        put(i, w);
        if constexpr (MARK) look(w);
    }
    if constexpr (MARK) {
        __shared__ int wave_marks[4];
        if ((tid & 63) == 0) wave_marks[tid >> 6] = mark;
        __syncthreads();
        if (amax < INFINITY && (wave_marks[0] | wave_marks[1] | wave_marks[2] | wave_marks[3])) scale = -scale;
    }
    if (tid == 0) *row_scale = scale;
}

template <bool MARK = false>
__device__ __forceinline__ void jl_row_to_f16(const float *__restrict__ X, _Float16 *__restrict__ A,
                                              float *__restrict__ row_scale, int rows, int k, int row) {
    typedef _Float16 jl_half4 __attribute__((ext_vector_type(4)));
    _Float16 *a = A + (int64_t)row * k;
    if (row >= rows) {
        for (int i = threadIdx.x * 4; i < k; i += 1024) *(jl_half4 *)(a + i) = jl_half4{0, 0, 0, 0};
        if (threadIdx.x == 0) row_scale[row] = 1.f;
        return;
    }
    const float *x = X + (int64_t)row * k;
    if (k <= 2048) jl_row_to_f16_held<2, MARK>(x, a, row_scale + row, k);
    else if (k <= 4096) jl_row_to_f16_held<4, MARK>(x, a, row_scale + row, k);
    else jl_row_to_f16_held<8, MARK>(x, a, row_scale + row, k);
}
