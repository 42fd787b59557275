// A patch of an image in whole vectors of four floats, as the convolutions on rectangles (ConvF32Rect, ConvF32Few) stage it: which of them a lane takes, and
// what becomes of one that reaches beside the image.
#pragma once
#include <hip/hip_runtime.h>

namespace bfuse {

// NU units for LANES lanes, one a load, up to sixteen loads under way at a time.
template <int NU, int LANES>
struct PatchUnits {
    static constexpr int NLD = (NU + LANES - 1) / LANES;         // loads
    static constexpr int JB = NLD < 16 ? NLD : 16;               // loads of a batch; the last one has fewer, unless
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
