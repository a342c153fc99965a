// Three-way bf16 splits of fp32 numbers for the bf16 matrix cores: x = h + m + l, 8
// significant bits each (gemm_split.hip has the arithmetic and its error).
#pragma once
#include "jas_common.hpp"

namespace jas {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// The three planes of eight fp32 values (slots 0..7 of a lane).  Each residual is one
// v_dot2_f32_bf16 of the packed pair with (-1, 0) or (0, -1): x - h, exact, without unpacking
// h (7 instructions per pair; widening and subtracting took 11).  The two constants stay in
// registers: given -1.0 as an inline constant the instruction takes it as an fp32 pattern.
// Exact for every x with 2^-110 <= |x| that does not round to infinity in bf16 (checked over
// random bit patterns of every exponent).
// SCALED: the planes of 2^16 x.  fp32 numbers end at 2^-149 and bf16 ones at 2^-133, so these are
// exact for subnormal x too, up to 2^111, for two more instructions per pair.
constexpr float SPLIT_SCALE = 0x1p16f, SPLIT_UNSCALE = 0x1p-16f;
template <bool SCALED = false>
__device__ __forceinline__ void split8(const float (&v)[8], u32x4 &h, u32x4 &m, u32x4 &l)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    unsigned c0 = 0x0000bf80u, c1 = 0xbf800000u;  // bf16 (-1, 0) and (0, -1)
    asm("" : "+s"(c0));
    asm("" : "+s"(c1));
    const bf16x2 m0 = __builtin_bit_cast(bf16x2, c0), m1 = __builtin_bit_cast(bf16x2, c1);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float x0 = SCALED ? v[2 * j] * SPLIT_SCALE : v[2 * j], x1 = SCALED ? v[2 * j + 1] * SPLIT_SCALE : v[2 * j + 1];
        const bf16x2 a = {(__bf16)x0, (__bf16)x1};
        const float r0 = __builtin_amdgcn_fdot2_f32_bf16(a, m0, x0, false);
        const float r1 = __builtin_amdgcn_fdot2_f32_bf16(a, m1, x1, false);
        const bf16x2 b = {(__bf16)r0, (__bf16)r1};
        const float q0 = __builtin_amdgcn_fdot2_f32_bf16(b, m0, r0, false);
        const float q1 = __builtin_amdgcn_fdot2_f32_bf16(b, m1, r1, false);
        h[j] = __builtin_bit_cast(unsigned, a);
        m[j] = __builtin_bit_cast(unsigned, b);
        l[j] = __builtin_bit_cast(unsigned, bf16x2{(__bf16)q0, (__bf16)q1});  // exact: at most 8 significant bits
    }
}

// largest magnitude of the operand values a lane has split
__device__ __forceinline__ void track_max(float &mx, const float (&x)[8])
{
#pragma unroll
    for (int j = 0; j < 8; j += 2) asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(mx) : "v"(x[j]), "v"(x[j + 1]));
}

// acc += a b over one 32-wide step, the six products above 2^-26 of it, small ones first
__device__ __forceinline__ floatx4 mfma_split(const bf16x8 (&a)[3], const bf16x8 (&b)[3], floatx4 acc)
{
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], b[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[1], acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[0], acc, 0, 0, 0);
}

} // namespace jas
