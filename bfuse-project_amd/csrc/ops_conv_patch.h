// A patch of an image in whole vectors of four floats, as the convolutions on rectangles (ConvF32Rect, ConvF32Few) stage it: which of them a lane takes.
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

}  // namespace bfuse
