// fp32 products on the matrix cores' bfloat16 instructions.
//
// A number is held as the sum of three bfloat16 numbers, its top 8 significant bits, the next 8 and the last 8: exactly, unless
// it is infinite, a NaN or so small (below 2^-110) that the last part is no bfloat16 number.  Of the nine products of two such
// sums the six largest are made -- each exact, as 8 bits times 8 bits are 16 --; what is left out is below 2^-24 of the product,
// 2^-25 on average.
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

// Two numbers' parts, a pair of bfloat16 numbers each.  Returns the last parts' bits, for split_inexact().  hi_mask is
// 0xffff0000 in a vector register: an instruction with a scalar operand takes twice as long.
__device__ __forceinline__ unsigned split2(float x0, float x1, unsigned hi_mask, unsigned &p0, unsigned &p1, unsigned &p2)
{
    const unsigned b0 = __builtin_bit_cast(unsigned, x0), b1 = __builtin_bit_cast(unsigned, x1);
    const float r0 = x0 - __builtin_bit_cast(float, b0 & hi_mask), r1 = x1 - __builtin_bit_cast(float, b1 & hi_mask);
    const unsigned c0 = __builtin_bit_cast(unsigned, r0), c1 = __builtin_bit_cast(unsigned, r1);
    const unsigned d0 = __builtin_bit_cast(unsigned, r0 - __builtin_bit_cast(float, c0 & hi_mask));
    const unsigned d1 = __builtin_bit_cast(unsigned, r1 - __builtin_bit_cast(float, c1 & hi_mask));
    p0 = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
    p1 = __builtin_amdgcn_perm(c1, c0, 0x07060302u);
    p2 = __builtin_amdgcn_perm(d1, d0, 0x07060302u);
    return d0 | d1;
}
__device__ __forceinline__ unsigned split4(split_f4 x, unsigned hi_mask, split_u2 (&p)[3])
{
    unsigned a, b, c, low = split2(x[0], x[1], hi_mask, a, b, c);
    p[0][0] = a; p[1][0] = b; p[2][0] = c;
    low |= split2(x[2], x[3], hi_mask, a, b, c);
    p[0][1] = a; p[1][1] = b; p[2][1] = c;
    asm volatile("" : "+v"(low));                    // (here: the compiler would keep every last part for later)
    return low;
}
__device__ __forceinline__ unsigned split8(const float (&x)[8], unsigned hi_mask, split_u4 (&p)[3])
{
    unsigned low = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned a, b, c;
        low |= split2(x[2 * i], x[2 * i + 1], hi_mask, a, b, c);
        p[0][i] = a; p[1][i] = b; p[2][i] = c;
    }
    asm volatile("" : "+v"(low));
    return low;
}
// Whether, by the last parts' bits, some number was not held exactly: bits below a bfloat16 number's, or an exponent of all
// ones (also where numbers above 2^17 meet by chance: the caller's exact way is right for any).
__device__ __forceinline__ bool split_inexact(unsigned low) { return (low & 0xffffu) != 0u || (low & 0x7f800000u) == 0x7f800000u; }

__device__ __forceinline__ split_f4 split_mfma(split_u4 a, split_u4 b, split_f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(split_b8, a), __builtin_bit_cast(split_b8, b), c, 0, 0, 0);
}

}  // namespace
}  // namespace cuvdia
