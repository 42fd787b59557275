// fp32 products on the bf16 matrix cores.
//
// x = p0 + p1 + p2 with p0 the nearest bf16 to x, p1 the nearest to x - p0 and p2 what is left: three times eight bits and two
// signs hold the 24 bits of an fp32 exactly.  Of the nine products of two such sums the three smallest (p1 q2, p2 q1, p2 q2: 2^-26
// of the product at most, 1e-8 of it in the mean) are left out.  The MFMA's products of two bf16 are exact, 32 of them are added
// to the accumulator with one rounding to nearest, and bf16 and fp32 denormals are kept (all of it as measured on the card).
//
// What the parts cannot hold:
//   * infinities and NaN, and finite values whose nearest bf16 is infinite (2^128 - 2^119 and up): x - p0 is then infinite or NaN,
//     and so is every result that x has a part in.  A kernel looks at its results and multiplies those that are not finite again
//     with the fp32 instructions, so that what comes out is what fp32 arithmetic gives;
//   * bits below 2^-133, bf16's smallest: those of values below 2^-109.  Beside a value of 2^-95 or more in the same row (column)
//     they are 2^-38 of it.  A kernel ors the leading parts of what each thread takes apart; where some are not zero and all lie
//     below 2^-95 (the three leading bits of every exponent zero) it does the tile again likewise.
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

// Two fp32 as three words of two bf16 each (lo in the low halves).
__device__ __forceinline__ void split2(float lo, float hi, unsigned& p0, unsigned& p1, unsigned& p2)
{
    p0 = pack_bf16(lo, hi);
    const float l1 = lo - __builtin_bit_cast(float, p0 << 16), h1 = hi - __builtin_bit_cast(float, p0 & 0xffff0000u);
    p1 = pack_bf16(l1, h1);
    const float l2 = l1 - __builtin_bit_cast(float, p1 << 16), h2 = h1 - __builtin_bit_cast(float, p1 & 0xffff0000u);
    p2 = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, h2), __builtin_bit_cast(unsigned, l2), 0x07060302u);   // their upper halves
}

__device__ __forceinline__ f32x4 mfma_bf16(u32x4 a, u32x4 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Whether the values whose leading parts were or-ed into `seen` are all below 2^-95 without all being zero.
__device__ __forceinline__ bool split_tiny(unsigned seen)
{
    return (seen & 0x7fff7fffu) != 0 && (seen & 0x70007000u) == 0;
}

// The products (part A[t] of one operand, part B[t] of the other); all but the last are 2^-8 and less of it.  Part 2 of B is done
// with first, part 1 next: their registers take the next columns' parts while part 0 is still in use.
struct SplitTerms {
    static constexpr int N = 6;
    static constexpr int A[N] = {0, 0, 1, 2, 1, 0}, B[N] = {2, 1, 1, 0, 0, 0};
};

}  // namespace bfuse
