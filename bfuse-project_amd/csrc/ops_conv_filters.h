// A operand of the convolutions whose waves have channel groups of 16 to themselves (Conv3x3F32Lds, ConvF32Lds): the filters of
// 16 TM output channels over one group, lane (i, q) ending up with filter row i's channels 4q .. 4q + 3, 4 T consecutive floats.
//
// Loaded as the lanes want them, a wave's load takes 16 bytes in each of 64 lines, and the CU's address unit 64 clocks for it:
// T such loads of every wave, 2300 clocks on the critical path of a 3 x 3 layer of four waves.  Here a load takes 64 consecutive
// bytes of each of 16 rows (16 clocks) straight into LDS, a place of the wave's own, and the lanes read their floats from
// there: T 128-bit reads.  Chunk c of a row lies at c ^ (row / 4) of its 64 bytes, so that the 16 lanes of a quarter of such a read meet no
// bank twice.  us alone, before and now: 64 -> 64 channels on 56 x 56 6.9 -> 5.4, 128 on 28 x 28 (32 output channels a workgroup) 9.0 -> 6.2.
// (Through registers and 128-bit LDS writes, which run at 80 B a clock: 5.6 and 6.8.)
#pragma once
#include <hip/hip_runtime.h>

#include "wave.h"

namespace bfuse {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int CI, int T, int TM>
struct FilterRows {
    static constexpr int BYTES = 1024 * T;      // LDS for 16 rows of 16 channels
    f32x4 w[TM][T];

    // The filters of row block tm on their way into `room` (BYTES): T loads.
    __device__ static __forceinline__ void request(const float* Wt, int co0, int ci0, int tm, unsigned char* room, int lane)
    {
        const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)(Wt + ((size_t)(co0 + 16 * tm) * CI + ci0) * T), 0, (15 * CI + 16) * T * 4, 0x00020000);
        const unsigned voff = (unsigned)((lane >> 2) * CI * T * 4 + ((lane & 3) ^ (lane >> 4)) * 16);
#pragma unroll
        for (int j = 0; j < T; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void*)(room + j * 1024), 16, voff, j * 64, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    }
    // They are here, with BEHIND loads of this wave on their way since, and go to registers: `room` is free again.  (The build counts
    // the loads behind the wait that says so.)
    template <int BEHIND>
    __device__ __forceinline__ void take(int tm, const unsigned char* room, int lane)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("s_waitcnt vmcnt(%0) ; loads into LDS have landed" : : "n"(BEHIND < 63 ? BEHIND : 63) : "memory");
#endif
        const int li = lane & 15, kq = lane >> 4;
#pragma unroll
        for (int j = 0; j < T; ++j) {
            const int c = kq * T + j;
            w[tm][j] = *reinterpret_cast<const f32x4*>(room + (c >> 2) * 1024 + li * 64 + ((c & 3) ^ (li >> 2)) * 16);
        }
        reads_done();
    }
    // This wave's LDS reads have ended: what they read may be written over, by a load too.
    __device__ static __forceinline__ void reads_done()
    {
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#endif
        __builtin_amdgcn_sched_barrier(0);
    }
};

// The same for images of at most four channels (ConvF32Few), whose MFMAs have four rows of the window at a tap, or four taps of the rows that are left, for
// their k: lane (i, q) gets, of filter row i, RPL rows of the window from row q RPL on, which are consecutive floats, and taps q, 4 + q .. of the rest (zeros past the last one).  16 rows
// are 16 CI KH KW consecutive floats; lanes behind them load the last ones again.  A workgroup comes here once and has one wave, so the loads are written by hand and
// everything that is under way is waited for.  (Through registers the 7 x 7 layer of 1024 images took 5 % longer: a wave has not enough of them.)
template <int CI, int KH, int KW, int TM>
struct FilterFloats {
    static constexpr int ROWS = CI * KH, RPL = ROWS / 4, LEFT = ROWS % 4 * KW, NLT = (LEFT + 3) / 4, NM = RPL * KW + NLT, N = ROWS * KW;
    static constexpr int SIZE = 16 * N * 4, LOADS = (SIZE + 1023) / 1024, BYTES = 1024 * LOADS;
    typedef __attribute__((address_space(3))) unsigned char lds_u8;
    float w[TM][NM];

    // The first 16 rows on their way into `room` (BYTES).
    __device__ static __forceinline__ void request(const float* Wt, int co0, int tm, unsigned char* room, int lane)
    {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const unsigned at = (unsigned)(lane * 16 + j * 1024);
            dma_load_lds_b128(j * 1024 + 1024 <= SIZE || at + 16 <= SIZE ? at : SIZE - 16, Wt + (size_t)(co0 + 16 * tm) * N, (unsigned)(unsigned long long)(lds_u8*)(room + j * 1024));
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __device__ __forceinline__ void pick(int tm, const float* row, int kq)
    {
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const int i = m - RPL * KW, k = 4 * RPL * KW + 4 * i + kq;
            w[tm][m] = i < 0 ? row[kq * RPL * KW + m] : row[k < N ? k : N - 1];
            if (i >= 0 && 4 * i + 3 >= LEFT) w[tm][m] = k < N ? w[tm][m] : 0.f;
        }
    }
    // All of them to registers, `room` is free again.
    __device__ __forceinline__ void take(const float* Wt, int co0, unsigned char* room, int lane)
    {
        const int li = lane & 15, kq = lane >> 4;
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            if (tm > 0) request(Wt, co0, tm, room, lane);
#if defined(__HIP_DEVICE_COMPILE__)
            asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
#endif
            pick(tm, reinterpret_cast<const float*>(room) + li * N, kq);
#if defined(__HIP_DEVICE_COMPILE__)
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#endif
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // Filters that are too many for that, as they lie in memory.
    __device__ __forceinline__ void load(const float* Wt, int co0, int lane)
    {
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) pick(tm, Wt + (size_t)(co0 + 16 * tm + (lane & 15)) * N, lane >> 4);
    }
};

}  // namespace bfuse
