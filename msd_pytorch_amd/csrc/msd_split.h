// fp32 products on the bf16 matrix cores without loss of precision.
//
// An fp32 value is exactly the sum of three bf16 values (8 + 8 + 8 bits of significand, each part
// rounded to nearest): v = h + m + l with |m| <= 2^-8 |v| and |l| <= 2^-16 |v|.  A product of two
// such values is then the six products h h', h m', m h', m m', h l', l h' (smallest first into an
// fp32 accumulator); what is left out, m l' + l m' + l l', is at most 2^-23 of the product, of
// either sign, 2^-26 of it on average: below what rounding every product of an fp32 chain costs.
// v_mfma_f32_16x16x32_bf16 does 512 multiply-adds per cycle and SIMD where v_mfma_f32_16x16x4_f32
// does 32 (measured: 18 and 33 cycles per instruction), so the six take 0.4 of the time of the fp32
// product, and unlike that one they leave the vector pipe free (two vector instructions fit beside
// each at no cost, beside the fp32 instruction none).
//
// Values are taken 2^24 times as large: the lowest bit of an fp32 number, 2^-149, is then 2^-125, a normal bf16 number,
// so that the sum is exact however small the value is.  Products come 2^48 times as large; where they are added to
// what has been summed before, the same instruction takes that back.  (Without it values below 2^-110 lost their low
// parts: products of values around 2^-122 were off by 1e-4 to 3e-3.)
//
// Values from 2^36 on (6.9e10), infinities and NaN are reported by split8: the sum of a few hundred products of such
// values might not fit.  Callers take v_mfma_f32_16x16x4_f32 for the product at hand, on the values as they are.
#pragma once

#include "msd_common.h"

namespace msd {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

struct Split8 {
    bf16x8_t p[3];                                // high, middle, low part
};

constexpr float kSplitScale = 0x1p24f;            // of a value, and what takes that of a product back
constexpr float kSplitUnit = 0x1p-48f;

// The parts of values that have been multiplied by kSplitScale.  Returns a sum that is not finite where one of them has
// to be taken whole: 2^68 times a high part of 2^60 or more is an infinity.
__device__ __forceinline__ float split8(const float (&v)[8], Split8 &s)
{
#pragma clang fp contract(off)                    // (the scale is multiplied once: as a part of each difference it costs more)
    typedef float f2_t __attribute__((ext_vector_type(2)));
    float bad = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const f2_t x{v[i], v[i + 1]};
        const bf16x2_t h = __builtin_convertvector(x, bf16x2_t);
        const f2_t hf = __builtin_convertvector(h, f2_t);
        const f2_t r{x[0] - hf[0], x[1] - hf[1]};
        const bf16x2_t m = __builtin_convertvector(r, bf16x2_t);
        const f2_t mf = __builtin_convertvector(m, f2_t);
        const f2_t q{r[0] - mf[0], r[1] - mf[1]};
        const bf16x2_t l = __builtin_convertvector(q, bf16x2_t);
        bad = __builtin_amdgcn_fdot2_f32_bf16(h, bf16x2_t{(__bf16)0x1p68f, (__bf16)0x1p68f}, bad, false);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            s.p[0][i + e] = h[e];
            s.p[1][i + e] = m[e];
            s.p[2][i + e] = l[e];
        }
    }
    return bad;
}
__device__ __forceinline__ bool taken_whole(float bad) { return !__builtin_isfinite(bad); }

// Whole values in the place of their parts: the upper and the lower half of their bits.
__device__ __forceinline__ void put_whole(const float (&v)[8], Split8 &s)
{
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t bits = __float_as_uint(v[i]);
        s.p[0][i] = __builtin_bit_cast(__bf16, (uint16_t)(bits >> 16));
        s.p[1][i] = __builtin_bit_cast(__bf16, (uint16_t)bits);
        s.p[2][i] = (__bf16)0.f;
    }
}
__device__ __forceinline__ float whole_value(__bf16 upper, __bf16 lower)
{
    return __uint_as_float((uint32_t)__builtin_bit_cast(uint16_t, upper) << 16 | __builtin_bit_cast(uint16_t, lower));
}

// acc += a b for the parts of a (rows, k) and b (k, columns).
typedef float f32x4_acc_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4_acc_t mfma_split(const bf16x8_t (&a)[3], const bf16x8_t (&b)[3], f32x4_acc_t acc, int step)
{
    constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, ib[6] = {0, 2, 1, 0, 1, 0};
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ia[step]], b[ib[step]], acc, 0, 0, 0);
}

}  // namespace msd
