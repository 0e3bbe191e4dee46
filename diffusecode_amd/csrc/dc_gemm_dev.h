// dc_gemm_dev.h -- device helpers shared by the phase-GEMM kernels
// (dc_gemm.hip: rows x columns, dc_fold.h: rows x mirrored column pairs).
#pragma once
#include "dc_internal.h"

namespace dc {

constexpr int SCH_FP32 = 0;
constexpr int SCH_BF16X3 = 1;
constexpr int SCH_FP16X2 = 2;
constexpr int SCH_FP16X3 = 3;
constexpr int SCH_FP32D = SCHEME_FP32_ACC64;
// FP32 operands on v_mfma_f32_16x16x4_f32 (FP32D: partial sums kept in FP64)
__host__ __device__ constexpr bool fp32ops(int s) { return s == SCH_FP32 || s == SCH_FP32D; }
// three products (hi.hi, hi.lo, lo.hi) with both sides split
__host__ __device__ constexpr bool split3(int s) { return s == SCH_BF16X3 || s == SCH_FP16X3; }
// FP16 operands (v_mfma_f32_16x16x32_f16)
__host__ __device__ constexpr bool f16ops(int s) { return s == SCH_FP16X2 || s == SCH_FP16X3; }

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int SCHEME>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (f16ops(SCHEME))
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
    else
        return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}
template <int SCHEME>
__device__ __forceinline__ f32x2 unpack2(uint32_t w) {
    if constexpr (f16ops(SCHEME))
        return __builtin_convertvector(__builtin_bit_cast(f16x2, w), f32x2);
    else
        return (f32x2){__builtin_bit_cast(float, w << 16), __builtin_bit_cast(float, w & 0xFFFF0000u)};
}

// Low FP16 halves of a split: given h = (f16(x), f16(y)) packed, returns
// (f16(x - h.x), f16(y - h.y)) packed.  x - h.x is exact in FP32, so each
// half is one rounding, as with a conversion of the FP32 difference; the
// mixed-precision FMAs take 2 instructions where unpacking h, subtracting
// and packing again takes 5.
__device__ __forceinline__ uint32_t lo_halves_f16(uint32_t h, float x, float y) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, -1.0, %1, %2 op_sel_hi:[0,1,0]\n\t"
        "v_fma_mixhi_f16 %0, -1.0, %1, %3 op_sel:[0,1,0] op_sel_hi:[0,1,0]"
        : "=&v"(r)
        : "v"(h), "v"(x), "v"(y));
    return r;
}

// Round the 64-bit phase to the 32-bit turn fraction used by sincos_turn.
__device__ __forceinline__ uint32_t phase_top(uint64_t p) { return (uint32_t)((p + 0x80000000ull) >> 32); }

__device__ __forceinline__ float2 cmul(float2 x, float2 y) {
    return make_float2(__builtin_fmaf(x.x, y.x, -x.y * y.y), __builtin_fmaf(x.x, y.y, x.y * y.x));
}
__device__ __forceinline__ float2 cis(uint64_t ph) {
    float c, s;
    sincos_turn(phase_top(ph), c, s);
    return make_float2(c, s);
}

// Damped FP16 operands.  exp(-B s^2) of a row or column leaves FP16's range (22
// bits above 2^-2, 65,504 at most) where B s^2 is large either way, so the
// operands carry exp(-(B - Bref) s^2) and the epilogue multiplies by exp(-Bref s^2).
// Bref is the least B of the slice's occupied atoms: the factors are at most
// 1 (s^2 >= 0, split_sq), and those that are small are so beside the term of that
// atom in the same sum.
constexpr float NO_B = 3.0e38f;            // least B of no atoms
__device__ __forceinline__ float damp_ref(float bmin) {
    const float b = bmin < NO_B ? bmin : 0.0f;
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, b)));   // uniform
}
// c exp(-bref (s + lo)) as a float and what is left of it (to 1e-11); lo: what a
// float leaves of s^2.  The factor is one for a whole row or column, and s^2 is for all
// atoms, so their rounding does not average out as that of the operands does.
// (24 members on 93 x 215 points, chi^2, which amplifies a common error of F by
// I / (I - T): 2.9e-6 with the factor in one float.)
__device__ __forceinline__ float2 damp_back2(float bref, float s, float lo, double c) {
    const double p = -1.44269504088896340736 * (double)bref * ((double)s + (double)lo), n = rint(fmax(-1000.0, fmin(1000.0, p)));
    const double x = (p - n) * 0.69314718055994530942;
    double e = 1.0 / 362880.0;             // exp(x), |x| <= 0.35: Taylor to x^9, 1e-11
    e = __builtin_fma(e, x, 1.0 / 40320.0);
    e = __builtin_fma(e, x, 1.0 / 5040.0);
    e = __builtin_fma(e, x, 1.0 / 720.0);
    e = __builtin_fma(e, x, 1.0 / 120.0);
    e = __builtin_fma(e, x, 1.0 / 24.0);
    e = __builtin_fma(e, x, 1.0 / 6.0);
    e = __builtin_fma(e, x, 0.5);
    e = __builtin_fma(e, x, 1.0);
    e = __builtin_fma(e, x, 1.0);
    const double d = ldexp(e * c, (int)n);
    const float h = (float)d;
    return make_float2(h, (float)(d - (double)h));
}
// the product of two such factors
__device__ __forceinline__ float2 mul2(float2 a, float2 b) {
    const float h = a.x * b.x;
    return make_float2(h, __builtin_fmaf(a.x, b.x, -h) + __builtin_fmaf(a.x, b.y, a.y * b.x));
}
// 2^-(bref sv), to FP32's rounding
__device__ __forceinline__ float damp_back(float bref, float sv) {
    const float p = bref * sv, lo = __builtin_fmaf(bref, sv, -p);
    return __builtin_amdgcn_exp2f(-p) * __builtin_fmaf(lo, -0.6931471805599453f, 1.0f);
}

// Packed planes hold one u32 (re | im << 16) per (row, atom): 16 words per
// row, the four 16-byte atom quads of a row XOR-swizzled by bits 2..3 of the
// row so that 16-byte accesses of the element builders (4 atom quads x 4 rows) and
// of the MFMA operand reads (16 rows, one quad) fall on distinct banks.
__device__ __forceinline__ int pk_off(int row, int quad) { return row * 16 + 4 * (quad ^ ((row >> 2) & 3)); }
}  // namespace dc
