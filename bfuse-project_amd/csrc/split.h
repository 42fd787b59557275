// fp32 products on the bf16 matrix cores.
//
// x = p0 + p1 + p2 with p0 the nearest bf16 to x, p1 the nearest to x - p0 and p2 what is left: three times eight bits and two
// signs hold the 24 bits of an fp32 exactly (the published three-part split of single precision over bfloat16).  Of the nine
// products of two such sums the three smallest (p1 q2, p2 q1, p2 q2) are left out: 0.06 u of the product in the mean of normal
// operands, u = 2^-24, but p1 q2 and p2 q1 reach u / 2 each where both values lie just above 1 + 2^-8 times a power of two (0.99 u
// together at 0x1.00fe8p0 squared; 3.5 % of normal pairs have more than u / 4).  The MFMA's products of two bf16 are exact; the
// accumulator is first cut off (towards minus infinity) at half a unit in the last place of the largest product, its exponents
// added and not normalised, then the sum is rounded once to nearest; bf16 and fp32 denormals are kept.  (As measured on the card:
// this model gives all bits of 40960 sums of one product.)  So a sum of one product is off by 3 u at most (2.3 u seen) where the
// fp32 instructions are off by one; a product by a power of two is exact, as its factor's other parts are zero.  Sums of many
// products are closer than theirs (ops_gemm_split.h).
//
// What the parts cannot hold:
//   * infinities and NaN, and finite values whose nearest bf16 is infinite (2^128 - 2^119 and up): x - p0 is then infinite or NaN,
//     and so is every result that x has a part in.  A kernel looks at its results and multiplies those that are not finite again
//     with the fp32 instructions, so that what comes out is what fp32 arithmetic gives;
//   * bits below 2^-133, bf16's smallest: those of values below 2^-109.  What is left for p2 then has bits in its lower half,
//     which is dropped.  A kernel ors all that was left for p2; if a lower half is not zero, it does the tile again likewise.
#pragma once
#include <hip/hip_runtime.h>

#include "wave.h"

namespace bfuse {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Lets the compiler know that an asm statement with a memory clobber (a barrier, BlockSync::raw) may read and write this LDS
// buffer: without it the buffer is memory that only the visible loads and stores touch, and they move across.
__device__ __forceinline__ void shared_with_asm(const void* lds)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : : "v"((unsigned)(unsigned long long)(const __attribute__((address_space(3))) void*)lds) : "memory");
#endif
}

// What is left of two fp32 without their part 0, as words of parts 1 and 2 (lo in the low halves).  `left` gets the bits of what is
// left for the last one.
__device__ __forceinline__ void split2_left(float l1, float h1, unsigned& p1, unsigned& p2, unsigned& left)
{
    p1 = pack_bf16(l1, h1);
    const unsigned l2 = __builtin_bit_cast(unsigned, l1 - __builtin_bit_cast(float, p1 << 16)), h2 = __builtin_bit_cast(unsigned, h1 - __builtin_bit_cast(float, p1 & 0xffff0000u));
    p2 = __builtin_amdgcn_perm(h2, l2, 0x07060302u);   // their upper halves
    left |= l2 | h2;
}

// Two fp32 as three words of two bf16 each.
__device__ __forceinline__ void split2(float lo, float hi, unsigned& p0, unsigned& p1, unsigned& p2, unsigned& left)
{
    p0 = pack_bf16(lo, hi);
    split2_left(lo - __builtin_bit_cast(float, p0 << 16), hi - __builtin_bit_cast(float, p0 & 0xffff0000u), p1, p2, left);
}

// One bit pattern at a time: a tree of ors over what is taken apart keeps all that was left in registers until its end.
__device__ __forceinline__ void gather_left(unsigned& left)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm("" : "+v"(left));
#endif
}

__device__ __forceinline__ f32x4 mfma_bf16(u32x4 a, u32x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The four groups of 16 lanes as the rows of a matrix, the components as its columns: transposed.
__device__ __forceinline__ void transpose_groups(f32x4& r)
{
#if defined(__HIP_DEVICE_COMPILE__)
    u32x4 u = __builtin_bit_cast(u32x4, r);
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(u[0], u[2], false, false)), b = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(u[1], u[3], false, false));
    const u32x2 c = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false)), d = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false));
    r = __builtin_bit_cast(f32x4, u32x4{c[0], c[1], d[0], d[1]});
#endif
}

// Whether one of the values taken apart is more than its three parts.
__device__ __forceinline__ bool split_inexact(unsigned left)
{
    return (left & 0xffffu) != 0;
}

// The products (part A[t] of one operand, part B[t] of the other); all but the last are 2^-8 and less of it.  Part 2 of B is done
// with first, part 1 next: their registers take the next columns' parts while part 0 is still in use.
struct SplitTerms {
    static constexpr int N = 6;
    static constexpr int A[N] = {0, 0, 1, 2, 1, 0}, B[N] = {2, 1, 1, 0, 0, 0};
};

}  // namespace bfuse
