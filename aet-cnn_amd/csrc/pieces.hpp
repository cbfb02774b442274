// Exact three-piece bf16 operands (see conv_split.hip for the arithmetic).
#pragma once

#include "conv_common.hpp"

namespace ach {

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// bf16 pair (lo = a, hi = b), rounded to nearest even
__device__ __forceinline__ unsigned pk_bf16(float a, float b)
{
    const v2f v = {a, b};
    const v2bf r = __builtin_convertvector(v, v2bf);
    return __builtin_bit_cast(unsigned, r);
}
__device__ __forceinline__ float bf_lo(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(unsigned u) { return __uint_as_float(u & 0xffff0000u); }

// Operands are split as kPieceUp * f: the last bit of any float, subnormals
// included, is then at least 2^-125, so no piece is below bf16's normal range
// (unscaled, the pieces of values under 2^-110 lost bits: 2.6e-6 instead of
// 4e-7 from 64 bits at 1e-35, 2.6e-4 at 1e-37; scaled 1.4e-7 at any magnitude).
// Sums of products are taken back with kSumDown, exact but for a result that
// is subnormal itself.  Values above 2^103 and sums above 2^80 come out
// non-finite and take the fp32 recomputation.
constexpr float kPieceUp = 0x1p24f, kSumDown = 0x1p-48f;

// eight floats -> three pieces of eight bf16 (kPieceUp * f = p[0] + p[1] + p[2] exactly)
__device__ __forceinline__ void split8(const float *f, v4u *p)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = f[2 * i] * kPieceUp, b = f[2 * i + 1] * kPieceUp;
        const unsigned h = pk_bf16(a, b);
        const float ra = a - bf_lo(h), rb = b - bf_hi(h);
        const unsigned m = pk_bf16(ra, rb);
        p[0][i] = h;
        p[1][i] = m;
        p[2][i] = pk_bf16(ra - bf_lo(m), rb - bf_hi(m));
    }
}

__device__ __forceinline__ v8bf as_bf(v4u v) { return __builtin_bit_cast(v8bf, v); }

// Whether a plan's sums are no further from 64 bits than the fp32 kernel's.
// Rounding errors of a chain of additions add up as squares: with the sum
// growing evenly, n roundings come to u = 1.8e-8 sqrt(n) of it.  In units of
// u^2 a chain of L products on the fp32 instructions is L (6.0e-7 for 1152,
// 128 -> 128 @ 32x32), or 0.45 to 0.5 L where every second input is a relu's
// zero (4.3e-7), and adding up parts is their number; a step of 16 products here is
// `mixed` or `relu`, as measured on long chains and a tenth more.
struct StepError {
    double mixed, relu;
};
inline bool no_more_error(const StepError &e, double steps, double parts, double fp32_products,
                          double fp32_parts)
{
    return e.mixed * steps + parts <= fp32_products + fp32_parts &&
           e.relu * steps + parts <= 0.45 * fp32_products + fp32_parts;
}

#define MFMA_BF(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)

}  // namespace ach
