// How the per-wave convolutions (Conv3x3F32Lds, ConvF32Lds, ConvF32Rect, ConvF32Few) load the patches that they stage, and which whole vectors of four floats
// a lane takes on rectangles, and what becomes of one that reaches beside the image.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "wave.h"

namespace bfuse {

// Whether the FLOATS floats that a patch's loads can reach are too many for a buffer: the place outside the image, byte 2^31 - 1, has to lie past its end.
// (Self-tests say so of small ones.)
template <long long FLOATS>
inline constexpr bool kFarPatch = FLOATS * 4 > 0x7fffffffLL;

// The patch's loads: a buffer with its own range check, or, for images of 2 GiB and more (of the channels of a group), a test of every float.
// Where a wait for the filters counts the loads behind them (FilterRows::take), all of these have to be made and to stay ahead of it, whatever the compiler
// knows of them.  So where the last one is used by some lanes only the pointer is opaque (a memory clobber orders nothing against a `__restrict__` argument: that load was
// moved behind the wait, into the condition), and where one tile has all rows so is the first (of two loads known to lie outside the image one was made).
template <long long FLOATS>
struct PatchSource {
    static constexpr bool FAR = kFarPatch<FLOATS>;
    using Index = std::conditional_t<FAR, long long, int>;
    using Place = std::conditional_t<FAR, long long, unsigned>;
    // How many loads are under way behind the filters' where LOADS were written down.
    template <int LOADS>
    using Behind = std::integral_constant<int, FAR ? 0 : LOADS>;

    // HIDDEN: the pointer is opaque.
    template <bool HIDDEN>
    __device__ static __forceinline__ auto open(const float* x)
    {
        if constexpr (HIDDEN) x = opaque_pointer(x);
        if constexpr (FAR) return x;
        else return __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, (int)(FLOATS * 4), 0x00020000);
    }
    // Float `at` of them, and a place outside the image.
    __device__ static constexpr __forceinline__ Place place(Index at) { return FAR ? (Place)at : (Place)(at * 4); }
    __device__ static constexpr __forceinline__ Place outside() { return FAR ? (Place)-4096 : (Place)0x7fffffff; }
    // N floats from there on; those outside are zeros.
    template <int N, class Source>
    __device__ static __forceinline__ auto load(Source from, Place at)
    {
        typedef float vec __attribute__((ext_vector_type(N)));
        vec v;
        if constexpr (FAR) {
#pragma unroll
            for (int e = 0; e < N; ++e) v[e] = (unsigned long long)(at + e) < (unsigned long long)FLOATS ? from[at + e] : 0.f;
        } else if constexpr (N == 4) v = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0));
        else if constexpr (N == 2) v = __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b64(from, at, 0, 0));
        else v[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(from, at, 0, 0));
        return v;
    }
};

// How many of a patch's loads are under way at a time beside a lane's filters: sixteen take 64 registers, and what their addresses need, out of 256.  (Eight where they would all
// be one batch are 5 % of the time: 12 x 12 of four channels at stride 2, 13 loads, 484 us and 509.)
constexpr int loads_beside(int filters, int loads) { return filters > 190 || (filters > 96 && loads >= 16) ? 8 : 16; }

// NU units for LANES lanes, one a load, up to MOST loads under way at a time.
template <int NU, int LANES, int MOST = 16>
struct PatchUnits {
    static constexpr int NLD = (NU + LANES - 1) / LANES;         // loads
    static constexpr int JB = NLD < MOST ? NLD : MOST;           // loads of a batch; the last one has fewer, unless
    static constexpr int NBATCH = (NLD + JB - 1) / JB;
    static constexpr bool WHOLE = NLD % JB == 0;
    // Whether load j (of NBATCH JB) brings a unit to the lane whose would be u; what one that does not would store lies past the patch.
    __host__ __device__ static constexpr bool there(int j, int u) { return NU % LANES == 0 ? WHOLE || j < NLD : u < NU; }
};

// Columns of a patch that begin at column ix0 of an image W wide: STEP, a multiple of four, times the tile's place in its row, less the padding P.
// A buffer load gives zeros float by float past the buffer's end, but none at all of a vector that begins before the buffer.  So the vector that begins before
// column 0 and has columns of the image is read from column 0, and moved; the others from where they begin.
template <int W, int P, int STEP>
struct PatchColumns {
    static_assert(STEP % 4 == 0, "the vectors of every tile of a row have the same place in their four floats");
    static constexpr int SHIFT = P % 4;
    // (Where the padding is wider than a tile, that is another vector of the next tile.)
    __host__ __device__ static constexpr bool moved(int ix0, int vi) { return SHIFT != 0 && ix0 < 0 && vi == (P <= STEP ? P / 4 : -ix0 / 4); }
    // The column that vector vi of a row is loaded from.
    __host__ __device__ static constexpr int from(int ix0, int vi) { return ix0 + 4 * vi + (moved(ix0, vi) ? SHIFT : 0); }
    // Its float e as it goes to LDS, of what came.  `inside`: no vector of the patch reaches beside the image.
    template <class V>
    __host__ __device__ static constexpr float at(const V& came, int e, int ix0, int vi, bool inside)
    {
        return inside || (unsigned)(ix0 + 4 * vi + e) < (unsigned)W ? moved(ix0, vi) && e >= SHIFT ? came[e - SHIFT >= 0 ? e - SHIFT : 0] : came[e] : 0.f;
    }
};

}  // namespace bfuse
