// fp32 products on the matrix cores' bfloat16 instructions.
//
// A number is held as the sum of three bfloat16 numbers (the triple-bfloat16 splitting of Henry, Tang and Heinecke, "Leveraging
// the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", 2019): the nearest one, the one nearest to
// what that leaves, and the rest, which has at most 7 bits: exactly, unless it is infinite, a NaN, so large that the nearest
// bfloat16 number is infinite, or so small (below 2^-110) that the rest is no bfloat16 number.  Of the nine products of two such
// sums the six largest are made -- each exact, as 8 bits times 8 bits are 16 --; what is left out is at most 2^-24 of the
// product, 2^-27.5 in the quadratic mean of uniform numbers, of either sign alike (parts cut off instead: up to 2^-21, 2^-24.7 in
// the mean, and always towards zero).  Products within 2^-7 of the largest number may overflow, as their first parts' do.
//
// What the matrix core does with them, measured: 8 products at a time, columns ascending, what lies more than 24 bits below the
// largest of the 8 cut off, of the sum so far towards minus infinity; the new sum to the nearest fp32 number.  (Numbers below the normal ones
// are kept, among the parts and in the sums.)  Hence the small products first: only the first parts' sum is rounded at its own size.
#pragma once
#include <hip/hip_runtime.h>

namespace cuvdia {
namespace {

typedef float split_f4 __attribute__((ext_vector_type(4)));
typedef unsigned split_u2 __attribute__((ext_vector_type(2)));
typedef unsigned split_u4 __attribute__((ext_vector_type(4)));
typedef __bf16 split_b8 __attribute__((ext_vector_type(8)));

// A lane's number for work that is seldom done: what is derived from it is not kept in registers meanwhile.
__device__ __forceinline__ int here(int lane)
{
    asm volatile("" : "+v"(lane));
    return lane;
}

// Two numbers to two bfloat16 ones, the nearest each.
__device__ __forceinline__ unsigned split_near(float x0, float x1)
{
    unsigned p;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(p) : "v"(x0), "v"(x1));
    return p;
}
// What such a pair leaves of its numbers, exactly.  (Constants in vector registers: an instruction with a scalar operand or one
// of its own takes twice as long.)
struct SplitConst {
    unsigned hi_mask, half;
    __device__ __forceinline__ SplitConst() { asm volatile("v_mov_b32 %0, 0xffff0000\n\tv_mov_b32 %1, 16" : "=&v"(hi_mask), "=v"(half)); }
};
__device__ __forceinline__ void split_rest(unsigned p, const SplitConst &k, float &x0, float &x1)
{
    x0 -= __builtin_bit_cast(float, p << k.half);
    x1 -= __builtin_bit_cast(float, p & k.hi_mask);
}
__device__ __forceinline__ unsigned split_last(float x0, float x1, unsigned &low)
{
    const unsigned d0 = __builtin_bit_cast(unsigned, x0), d1 = __builtin_bit_cast(unsigned, x1);
    low |= d0 | d1;
    return __builtin_amdgcn_perm(d1, d0, 0x07060302u);
}
// Two numbers' parts, a pair of bfloat16 numbers each; the last parts' bits are added to low, for split_inexact.
__device__ __forceinline__ void split2(float x0, float x1, const SplitConst &k, unsigned &p0, unsigned &p1, unsigned &p2, unsigned &low)
{
    p0 = split_near(x0, x1);
    split_rest(p0, k, x0, x1);
    p1 = split_near(x0, x1);
    split_rest(p1, k, x0, x1);
    p2 = split_last(x0, x1, low);
}
__device__ __forceinline__ unsigned split4(split_f4 x, const SplitConst &k, split_u2 (&p)[3])
{
    unsigned low = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        unsigned a, b, c;
        split2(x[2 * i], x[2 * i + 1], k, a, b, c, low);
        p[0][i] = a; p[1][i] = b; p[2][i] = c;
    }
    asm volatile("" : "+v"(low));                    // (here: the compiler would keep every last part for later)
    return low;
}
__device__ __forceinline__ unsigned split8(const float (&x)[8], const SplitConst &k, split_u4 (&p)[3])
{
    unsigned low = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned a, b, c;
        split2(x[2 * i], x[2 * i + 1], k, a, b, c, low);
        p[0][i] = a; p[1][i] = b; p[2][i] = c;
    }
    asm volatile("" : "+v"(low));
    return low;
}
// Whether some number was not held exactly, by its wave's lanes' last parts: bits below a bfloat16 number's, or a NaN.  low: their
// bits; last(i), i < N: four pairs of them, asked for only where the exponents make up all ones, as those of numbers on both sides of
// 2^17 do together.
template <int N, class Last>
__device__ __forceinline__ bool split_inexact(unsigned low, Last &&last)
{
    if (__builtin_expect(!__any((low & 0xffffu) != 0u || (low & 0x7f800000u) == 0x7f800000u), 1)) return false;
    unsigned bad = low & 0xffffu;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const split_u4 pairs = last(i);
#pragma unroll
        for (int j = 0; j < 4; ++j) bad |= ((pairs[j] & 0x7f807f80u) + 0x00800080u) & 0x80008000u;
    }
    return __any(bad != 0u);
}

__device__ __forceinline__ split_f4 split_mfma(split_u4 a, split_u4 b, split_f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(split_b8, a), __builtin_bit_cast(split_b8, b), c, 0, 0, 0);
}

}  // namespace
}  // namespace cuvdia
