// split_bf16.h -- fp32 products on the bf16 matrix cores of gfx950, without
// giving up fp32 precision.
//
// x = hi + mid + lo with hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi -
// mid), each rounded to nearest: 3 x 8 bits hold the 24 bits of an fp32
// significand, so the sum is x itself, down to bf16's smallest number, 2^-133.
// fp32's is 2^-149: operands are multiplied by 2^16 (kSplitScale) as they are
// split, so that every fp32 number below 2^111 is split exactly, denormal ones
// too (the matrix core keeps denormal operands and sums, measured), and the
// results carry 2^32.  A product a*b is then
//   lo*hi' + hi*lo' + mid*mid' + mid*hi' + hi*mid' + hi*hi'
// with each part product exact in the matrix core; the three left out are at
// most 2^-24 |a b| together, one fp32 rounding (mid up to 2^-8 of x, lo up to
// 2^-17), and mostly far below it.  The small terms are added first.
// v_mfma_f32_32x32x16_bf16 does 8 times the work of v_mfma_f32_32x32x2f32 per
// instruction in half its time (8 against 16 passes), so six of them are 2.67
// times as fast, and they round the accumulator 6 times per 16 products where
// the fp32 instruction does it 8 times.  Measured against float64 (relative
// 2-norm error, N(0,1) operands): K = 64 1.1e-7 (fp32 instruction 1.4e-7),
// K = 4096 1.0e-6 (1.2e-6); U(0,1): K = 4096 5.3e-7 (8.6e-7).
//
// The matrix core rounds down, not to nearest, what it shifts out when it
// lines a sum's terms up: -0.004 ulp of the sum per instruction, and up to a
// whole ulp where the accumulator is the smaller term (measured over random
// operands).  That is far below the rounding of one element, but it has one
// sign, so sums over many elements (a bias gradient over 8192 rows) would
// collect it.  So a kernel gives each row and each column a sign (sign_of),
// contracts the signed operands and takes the sign off the result: the
// offset of neighbouring elements then differs in sign and cancels in sums.
// Measured at 4096^3, sum over the rows of a column, relative error: fp32
// instruction 1.1e-6, split 1.3e-5, split with signs 9.5e-7.
//
// What the split cannot carry is caught by the kernels that use it and
// computed again with the fp32 instruction: infinities, values from 2^111 on
// and sums from 2^96 on (a part or its remainder is infinite or NaN, so an
// accumulator that holds it is not finite).
//
// Operands of v_mfma_f32_32x32x16_bf16: lane l holds row (or column) l % 32
// and the 8 contraction elements of its half l / 32, as four packed pairs.
// Which elements those are only has to agree between A and B.
#pragma once

#include <hip/hip_runtime.h>

#include "mfma.h"

namespace ember {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 0x1p16f;

// The sign bit of row or column i: the top bit of i times 2^32 / golden ratio,
// which alternates evenly over every stride of i.
__device__ __forceinline__ unsigned sign_of(int i)
{
    return ((unsigned)i * 0x9E3779B9u) & 0x80000000u;
}
__device__ __forceinline__ unsigned float_bits(float x)
{
    return __builtin_bit_cast(unsigned, x);
}
__device__ __forceinline__ float flip(float x, unsigned sign)
{
    return __builtin_bit_cast(float, __builtin_bit_cast(unsigned, x) ^ sign);
}

// Two floats to packed bf16, rounded to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ unsigned pack_bf16(float x0, float x1)
{
    const f32x2 v = {x0, x1};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

// The parts of a pair: h, m, l are the packed hi, mid and lo.
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned &h, unsigned &m, unsigned &l)
{
    h = pack_bf16(x0, x1);
    x0 -= __builtin_bit_cast(float, h << 16);
    x1 -= __builtin_bit_cast(float, h & 0xffff0000u);
    m = pack_bf16(x0, x1);
    x0 -= __builtin_bit_cast(float, m << 16);
    x1 -= __builtin_bit_cast(float, m & 0xffff0000u);
    l = pack_bf16(x0, x1);
}

// Eight floats as the three parts of one operand.
struct Split8 {
    u32x4 part[3];  // hi, mid, lo
};

__device__ __forceinline__ Split8 split8(const float *v)
{
    Split8 s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned h, m, l;
        split_pair(v[2 * i], v[2 * i + 1], h, m, l);
        s.part[0][i] = h;
        s.part[1][i] = m;
        s.part[2][i] = l;
    }
    return s;
}

__device__ __forceinline__ f32x16 mfma_32x32x16(u32x4 a, u32x4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}

// Term t of a * b over 16 contraction elements; terms 0 to 4 are the small
// ones, 5 is hi * hi.
__device__ __forceinline__ void mfma_split_term(int t, const Split8 &a, const Split8 &b, f32x16 &c)
{
    constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
    c = mfma_32x32x16(a.part[pa[t]], b.part[pb[t]], c);
}

}  // namespace ember
