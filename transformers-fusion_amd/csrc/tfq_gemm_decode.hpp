// Operand types and the decode of packed codes to bf16 operands, shared by the prefill tile kernels
// (tfq_gemm.hip: weights rounded to bf16; tfq_gemm_exact.hip: integer operands).
#pragma once

#include "tfq_internal.hpp"

namespace tfq {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

__device__ __forceinline__ uint32_t bf16_rne(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}

// byte B of a dword as float (v_cvt_f32_ubyteB); written as an instruction because the optimizer
// otherwise rebuilds every nibble with a bit-field extract of its own, two operations per weight
template <int B>
__device__ __forceinline__ float ubyte_to_float(uint32_t v) {
    float f;
    if constexpr (B == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(f) : "v"(v));
    else if constexpr (B == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(f) : "v"(v));
    else if constexpr (B == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(f) : "v"(v));
    else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(f) : "v"(v));
    return f;
}

// one code dword (nibble t = weight t) -> eight bf16 weights in k order: 7 + 8 + 4 operations.
// (v >> 4 t) & 0x000F000F | 0x64006400 is the pair of binary16 numbers 1024 + n_t, 1024 + n_(t+4), exactly; the
// multiply-add reads either half as binary16 (v_fma_mix_f32) and takes c - 1024 a as its addend.  For the
// symmetric formats (a binary16 scale, c = -8 a or -128 a) that addend is exact in fp32 and a n + c is rounded
// once, to the same bits as a (float) n + c; for the affine formats it carries one rounding of its own, 2^-14
// of a, far below the bf16 rounding of the weight that follows.
// (M = 0x000F000F and C = 0x64006400 come in registers, so that (x & M) | C is one v_and_or_b32.)
__device__ __forceinline__ uint4 decode8(uint32_t v, float a, float c, uint32_t M, uint32_t C) {
    const float c2 = __builtin_fmaf(-1024.0f, a, c);
    const f16x2_t p0 = __builtin_bit_cast(f16x2_t, (v & M) | C), p1 = __builtin_bit_cast(f16x2_t, ((v >> 4) & M) | C);
    const f16x2_t p2 = __builtin_bit_cast(f16x2_t, ((v >> 8) & M) | C), p3 = __builtin_bit_cast(f16x2_t, ((v >> 12) & M) | C);
    uint4 o;
    o.x = pack_bf16(__builtin_fmaf(a, (float)p0.x, c2), __builtin_fmaf(a, (float)p1.x, c2));
    o.y = pack_bf16(__builtin_fmaf(a, (float)p2.x, c2), __builtin_fmaf(a, (float)p3.x, c2));
    o.z = pack_bf16(__builtin_fmaf(a, (float)p0.y, c2), __builtin_fmaf(a, (float)p1.y, c2));
    o.w = pack_bf16(__builtin_fmaf(a, (float)p2.y, c2), __builtin_fmaf(a, (float)p3.y, c2));
    return o;
}

// the same for an 8-bit code kept as two nibble planes (dword `lo`: low nibbles of codes 0..7, `hi`: high
// nibbles): the planes are merged to bytes first, 6 + 8 + 8 + 4 operations
__device__ __forceinline__ uint4 decode8x2(uint32_t lo, uint32_t hi, float a, float c) {
    const uint32_t ev = ((hi & 0x0F0F0F0Fu) << 4) | (lo & 0x0F0F0F0Fu);  // codes 0,2,4,6 as bytes
    const uint32_t od = (hi & 0xF0F0F0F0u) | ((lo >> 4) & 0x0F0F0F0Fu);  // codes 1,3,5,7
    uint4 o;
    o.x = pack_bf16(__builtin_fmaf(a, ubyte_to_float<0>(ev), c), __builtin_fmaf(a, ubyte_to_float<0>(od), c));
    o.y = pack_bf16(__builtin_fmaf(a, ubyte_to_float<1>(ev), c), __builtin_fmaf(a, ubyte_to_float<1>(od), c));
    o.z = pack_bf16(__builtin_fmaf(a, ubyte_to_float<2>(ev), c), __builtin_fmaf(a, ubyte_to_float<2>(od), c));
    o.w = pack_bf16(__builtin_fmaf(a, ubyte_to_float<3>(ev), c), __builtin_fmaf(a, ubyte_to_float<3>(od), c));
    return o;
}

// slope of the line that stands for the companded 8-bit grid in a matmul (level j ~ (j - 127.5) * gain,
// within 7.5e-5 relative of tanh(0.02 t) / tanh(0.02), src/codec/block_codec.cpp:224-237); the decode
// entry points use the exact table
constexpr float kComp8Line = 1.0000742443371564f / 127.5f;

// (a, c) of group g (0..7) of a block from its 16-byte header: weight = a * code + c
template <int FMT>
__device__ __forceinline__ void group_coeffs(uint4 h, int g, float& a, float& c) {
    if constexpr (FMT == TFQ_Q_G_4 || FMT == TFQ_Q_G_3) {
        const uint64_t scs = (uint64_t)h.x | ((uint64_t)(h.y & 0xFFFFu) << 32);
        const uint64_t mcs = (uint64_t)(h.y >> 16) | ((uint64_t)h.z << 16);
        const float sc = (float)(uint32_t)((scs >> (6 * g)) & 63u);
        const float mc = (float)((int)((mcs >> (6 * g)) & 63u) - 32);
        a = half_fast(h.w & 0xFFFFu) * sc * (FMT == TFQ_Q_G_4 ? 1.0f / 15.0f : 1.0f / 7.0f);
        c = -(half_fast(h.w >> 16) * mc);
    } else {
        // eight fp16 scales; the code is stored with an offset: 8 (4-bit), 128 (8-bit), 127.5 (companded grid)
        const uint32_t hw[4] = {h.x, h.y, h.z, h.w};
        a = half_fast((hw[g >> 1] >> (16 * (g & 1))) & 0xFFFFu);
        if constexpr (FMT == TFQ_B32S4) c = -8.0f * a;
        else if constexpr (FMT == TFQ_B32S8) c = -128.0f * a;
        else { a *= kComp8Line; c = -127.5f * a; }
    }
}

}  // namespace

}  // namespace tfq
