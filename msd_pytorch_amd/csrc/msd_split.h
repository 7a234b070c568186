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
// Values that have no such sum (infinities, NaN, and the few finite ones above 3.39e38, which round
// to an infinity) give a NaN in the rest of the split: callers look at that and take
// v_mfma_f32_16x16x4_f32 for the product at hand (split_any keeps the parts addable: h + m + l is the value).
#pragma once

#include "msd_common.h"

namespace msd {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

struct Split8 {
    bf16x8_t p[3];                                // high, middle, low part
};

// Returns a sum that is NaN where a value cannot be split.
__device__ __forceinline__ float split8(const float (&v)[8], Split8 &s)
{
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
        bad = __builtin_amdgcn_fdot2_f32_bf16(l, bf16x2_t{(__bf16)1.f, (__bf16)1.f}, bad, false);
#pragma unroll
        for (int e = 0; e < 2; e++) {
            s.p[0][i + e] = h[e];
            s.p[1][i + e] = m[e];
            s.p[2][i + e] = l[e];
        }
    }
    return bad;
}

// The parts of any value: those of a value that is not finite are itself and zeros, the high part is cut
// off, not rounded, so that it stays finite where the value is.
__device__ __forceinline__ void split_any(const float (&v)[8], Split8 &s)
{
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float h = v[i] != v[i] ? v[i] : __uint_as_float(__float_as_uint(v[i]) & 0xffff0000u);
        const bool finite = (__float_as_uint(h) & 0x7f800000u) != 0x7f800000u;
        const float r = finite ? v[i] - h : 0.f;
        const float m = __uint_as_float(__float_as_uint(r) & 0xffff0000u);
        s.p[0][i] = (__bf16)h;
        s.p[1][i] = (__bf16)m;
        s.p[2][i] = (__bf16)(r - m);
    }
}

// acc += a b for the parts of a (rows, k) and b (k, columns).
typedef float f32x4_acc_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4_acc_t mfma_split(const bf16x8_t (&a)[3], const bf16x8_t (&b)[3], f32x4_acc_t acc, int step)
{
    constexpr int ia[6] = {2, 0, 1, 1, 0, 0}, ib[6] = {0, 2, 1, 0, 1, 0};
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ia[step]], b[ib[step]], acc, 0, 0, 0);
}

}  // namespace msd
