// Convolution of images of at most four channels: the implicit GEMM of ConvF32Rect on a tile of TH output rows x 16 TWB output columns, one
// wave, whose MFMAs' four k are rows of the window instead of channels.
//
// The first layers of the example networks (three channels) have a small patch, many taps and more results than anything else:
//   * a window is CI KH rows of KW taps.  Each group of 16 lanes has a quarter of its rows, one tap of them at an MFMA; the taps of up to three rows that are left are dealt
//     out singly.  7 x 7 on RGB is 37 MFMAs for 16 pixels and channels, with the channels as k (the fourth of them zeros) it was 49;
//   * so the patch lies in LDS as it does in memory, rows of whole 16-byte vectors, and is written a vector at a time where [position][channel] took four
//     writes; the filters' rows are consecutive floats as well (FilterFloats);
//   * with TWB columns a lane a wave writes rows of 64 TWB bytes, 16 bytes a lane for four.  Results of one lane to a column, 64 bytes of a row that often
//     begins inside a line, are what bounds 3 x 3 layers (299 x 299 at stride 2, 2.9 GB of results: 1338 us with one column, 1267 with two, 1108 with four); 7 x 7 is bound by its MFMAs
//     and 64 columns leave more of them idle (112 columns: 2530 us with four, 2109 with one).  LINES: results larger than the
//     last-level cache whose rows are whole 64-byte pieces are written past the caches: 64 channels on 112 x 112, 256 images, 256 -> 183 us; with pieces of lines it is
//     the other way round (149 columns 1105 -> 1549);
//   * a sum is two halves, added up at the end: as one it is off by 1.00 - 1.02 times what the sum over taps of all channels was (2-norm), as two by 0.75 times; 3 % of
//     the time of 7 x 7, none elsewhere.
//
// us, with the channels as k, every float staged by itself and filters as the lanes want them (ConvF32Rect as it was), and now: 7 x 7 on 1024 RGB images of 224 x 224 3371 -> 2154, on one 8.75 -> 5.72, with the LayerNorm
// 12.2 -> 8.2, 3 x 3 at stride 2 on 1024 of 299 x 299 1484 -> 985.  (With filters through LDS and 32 channels a wave alone 2688, 7.26, 10.5 and 1338.)
#pragma once
#include <hip/hip_runtime.h>

#include "dispatch.h"
#include "ops_conv_filters.h"
#include "ops_conv_patch.h"
#include "wave.h"

namespace bfuse {

template <int CI_, int CO_, int H_, int W_, int KH_, int KW_, int S_, int P_, int BM_, int TH_, int TWB_, int NIMG_ = 1, bool LINES_ = false, bool SLIM_ = false>
struct ConvF32Few {
    static constexpr bool MATRIX_CORES = true;   // the inner loop is a stream of MFMAs (what the fusion chooser asks)
    static constexpr int CI = CI_, CO = CO_, H = H_, W = W_, KH = KH_, KW = KW_, S = S_, P = P_, BM = BM_, TH = TH_, TWB = TWB_, NIMG = NIMG_;
    static constexpr bool LINES = LINES_;
    static constexpr int OH = (H - KH + 2 * P) / S + 1, OW = (W - KW + 2 * P) / S + 1;
    static_assert(!LINES || OW % 16 == 0, "rows of whole pieces of lines");
    static constexpr int HW = H * W, OHW = OH * OW;
    static constexpr int TM = BM / 16;
    static constexpr int NTX = (OW + 16 * TWB - 1) / (16 * TWB), NTY = (OH + TH - 1) / TH, NPT = NTX * NTY;
    static constexpr int PR = (TH - 1) * S + KH, PC = ((16 * TWB - 1) * S + KW + 3) / 4 * 4;   // patch rows / columns, whole vectors of four
    using Filters = FilterFloats<CI, KH, KW, TM>;
    static constexpr int RPL = Filters::RPL, NLT = Filters::NLT, NM = Filters::NM, LEFT = Filters::LEFT, HALF = (NM + 1) / 2;
    // 16-channel blocks and rows that are summed up at a time, and the 16-pixel blocks of these
    static constexpr int TMP = SLIM_ ? 1 : TM, THP = !SLIM_ ? TH : NM > 72 ? 1 : TH % 4 == 0 ? 4 : TH, PB = THP * TWB;
    // The filters come to the registers through the wave's tile, before the patch is staged, where they are not much more than the patch.
    static constexpr bool TURNED = CI * KH * KW <= 160;
    static constexpr int PATCH_BYTES = CI * PR * PC * 4;
    static constexpr int TILE_BYTES = TURNED && Filters::BYTES > PATCH_BYTES ? Filters::BYTES : PATCH_BYTES;
    static constexpr int NVR = PC / 4;                  // vectors of a patch row
    static constexpr int NU = CI * PR * NVR;            // staging units (channel, row, vector)
    using Units = PatchUnits<NU, 64, (!SLIM_ ? loads_beside(NM * TM, (NU + 63) / 64) : NM > 72 ? 4 : 8)>;
    using Columns = PatchColumns<W, P, 16 * TWB * S>;
    using Source = PatchSource<(long long)CI * HW>;
    static constexpr int NLD = Units::NLD;              // wave-level loads
    static_assert(CI >= 1 && CI <= 4 && CO % BM == 0 && BM % 16 == 0, "channels");
    static_assert(S >= 1 && OH >= 1 && OW >= 1 && TH >= 1 && (PR * PC + KW) * 4 < 65536, "shape; offsets of rows and taps are 16-bit immediates");

    static constexpr int NCT = CO / BM;
    static_assert(NIMG >= 1 && (long long)NPT * NCT * NIMG < (1LL << 31), "grid size");
    static constexpr Dims3 GRID{NPT * NCT * NIMG, 1, 1};
    static constexpr Dims3 BLOCK{64, 1, 1};
    static constexpr int THREADS = 64;
    static constexpr bool HAS_BARRIERS = false;

    struct Smem {
        __attribute__((aligned(16))) unsigned char t[TILE_BYTES];
    };

    // Workgroup id -> (pixel tile of the batch, output-channel tile), as ConvF32Rect
    __device__ static __forceinline__ void tile_of(int vblock, int& pt, int& ct)
    {
        constexpr int NPTB = NPT * NIMG, PER_XCD = NPTB / 8, FULL = 8 * PER_XCD * NCT;
        if (vblock < FULL) {
            const int xcd = vblock & 7, slot = vblock >> 3;
            pt = xcd * PER_XCD + slot / NCT;
            ct = slot % NCT;
        } else {
            const int rem = vblock - FULL;
            pt = 8 * PER_XCD + rem / NCT;
            ct = rem % NCT;
        }
    }

    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync)
    {
        const float* __restrict__ X = static_cast<const float*>(I);
        const float* __restrict__ Wt = static_cast<const float*>(F);
        float* __restrict__ Y = static_cast<float*>(O);
        int pt, ct;
        tile_of(vblock, pt, ct);
        if constexpr (NIMG > 1) {
            const int img = pt / NPT;
            pt -= img * NPT;
            X += (size_t)img * CI * HW;
            Y += (size_t)img * CO * OHW;
        }
        const int co0 = ct * BM;
        const int oy0 = (pt / NTX) * TH, ox0 = (pt % NTX) * 16 * TWB;   // first output row / column of the tile
        const int iy0 = oy0 * S - P, ix0 = ox0 * S - P;           // image row / column of patch position (0, 0)
        const int lane = tid & 63, li = lane & 15, kq = lane >> 4;
        unsigned char* const tile = sm.t;

        Filters filters;
        if constexpr (TURNED) Filters::request(Wt, co0, 0, tile, lane);

        // Stage the patch, [channel][row][PC floats]: the lanes take its vectors in turn, which follow each other in LDS.  A vector of a row outside the image is
        // read past the buffer's end; floats beside the image are made zeros (PatchColumns).
        const auto xr = Source::template open<false>(X);
        const bool inside = ix0 >= 0 && ix0 + PC <= W;          // no vector reaches beside the image
        constexpr int JB = Units::JB;
        if constexpr (!TURNED) filters.load(Wt, co0, lane);
        else if constexpr (NLD > JB) filters.take(Wt, co0, tile, lane);
#pragma unroll 1
        for (int j0 = 0; j0 < NLD; j0 += JB) {
            f32x4 v[JB];
#pragma unroll
            for (int jj = 0; jj < JB; ++jj) {
                const int u = (j0 + jj) * 64 + lane, r = u / NVR, vi = u % NVR, c = r / PR, iy = iy0 + r - c * PR;
                v[jj] = Source::template load<4>(xr, iy >= 0 && iy < H && u < NU ? Source::place((typename Source::Index)c * HW + iy * W + Columns::from(ix0, vi)) : Source::outside());
            }
            if constexpr (NLD <= JB && TURNED) filters.take(Wt, co0, tile, lane);
            if (!inside) {
#pragma unroll
                for (int jj = 0; jj < JB; ++jj) {
                    const int u = (j0 + jj) * 64 + lane;
                    const f32x4 f = v[jj];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[jj][e] = Columns::at(f, e, ix0, u % NVR, false);
                }
            }
#pragma unroll
            for (int jj = 0; jj < JB; ++jj) {
                const int u = (j0 + jj) * 64 + lane;
                if (Units::there(j0 + jj, u)) *reinterpret_cast<f32x4*>(tile + u * 16) = v[jj];
            }
        }

        // Where this lane's rows of the window begin for its column, and its taps of the rows that are left.
        // (A quarter that stays in one channel has its rows one after the other, a constant apart.)
        constexpr bool RUN = RPL > 0 && KH % (RPL > 0 ? RPL : 1) == 0;
        const unsigned char* row[RPL > 0 && !RUN ? RPL : 1];
        const unsigned char* last[NLT > 0 ? NLT : 1];
        const auto at = [&](int r, int kw) { return tile + ((r / KH * PR + r % KH) * PC + kw + li * S * TWB) * 4; };
#pragma unroll
        for (int r = 0; r < (RUN ? 1 : RPL); ++r) row[r] = at(kq * RPL + r, 0);
#pragma unroll
        for (int i = 0; i < NLT; ++i) {
            const int t = 4 * i + kq < LEFT ? 4 * i + kq : 0;
            last[i] = at(4 * RPL + t / KW, t % KW);
        }
        auto value = [&](int m, int y0, int pb) {
            const unsigned char* const from = m < RPL * KW ? row[RUN || m / KW >= RPL ? 0 : m / KW] + ((RUN ? m / KW * PC : 0) + m % KW) * 4 : last[m - RPL * KW >= 0 ? m - RPL * KW : 0];
            const float f = *reinterpret_cast<const float*>(from + ((y0 + pb / TWB) * PC + pb % TWB) * S * 4);
            return m == NM - 1 && LEFT % 4 != 0 && kq >= LEFT % 4 ? 0.f : f;
        };
        typedef float cols __attribute__((ext_vector_type(TWB), aligned(4)));
        const int ox = ox0 + li * TWB;
#pragma unroll
        for (int pass = 0; pass < TM / TMP * (TH / THP); ++pass) {
            const int t0 = pass / (TH / THP) * TMP, y0 = pass % (TH / THP) * THP;
#if defined(__HIP_DEVICE_COMPILE__)
            if (pass > 0) asm volatile("" : : : "memory");   // the patch is read again, not kept
#endif
            f32x4 acc[2][TMP][PB];                              // the sums of the first and of the second half
            // read the next operands while these multiply
            float b[2][PB];
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) b[0][pb] = value(0, y0, pb);
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                if (m + 1 < NM) {
#pragma unroll
                    for (int pb = 0; pb < PB; ++pb) b[(m + 1) & 1][pb] = value(m + 1, y0, pb);
                }
#pragma unroll
                for (int tm = 0; tm < TMP; ++tm)
#pragma unroll
                    for (int pb = 0; pb < PB; ++pb) {
                        f32x4& sum = acc[m >= HALF][tm][pb];
                        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(filters.w[t0 + tm][m], b[m & 1][pb], m % HALF == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : sum, 0, 0, 0);
                    }
            }
            // lane (j = column of the tile row, rg) owns output channels 4 rg + v of a block
#pragma unroll
            for (int tm = 0; tm < TMP; ++tm)
#pragma unroll
                for (int y = 0; y < THP; ++y)
                    if (oy0 + y0 + y < OH) {
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            float* const to = Y + (size_t)(co0 + (t0 + tm) * 16 + 4 * kq + v) * OHW + (oy0 + y0 + y) * OW + ox;
                            cols c;
#pragma unroll
                            for (int b = 0; b < TWB; ++b) c[b] = NM > 1 ? acc[0][tm][y * TWB + b][v] + acc[1][tm][y * TWB + b][v] : acc[0][tm][y * TWB + b][v];
                            if (ox + TWB <= OW) {
                                if constexpr (LINES) __builtin_nontemporal_store(c, reinterpret_cast<cols*>(to));
                                else *reinterpret_cast<cols*>(to) = c;
                            } else {
#pragma unroll
                                for (int b = 0; b + 1 < TWB; ++b)
                                    if (ox + b < OW) to[b] = c[b];
                            }
                        }
                    }
        }
    }
};

// (see Slim) Sixteen channels and four rows at a time, or one beside many taps, and fewer loads under way: 32 channels with 64 columns of two rows, or 16 with
// eight rows, are 128 or 64 registers of sums, with which 3 x 3 layers (169 in all) and larger filters do not fit beside ten waves.  The patch is read again for each.
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int BM, int TH, int TWB, int NIMG, bool LINES>
struct SlimOf<ConvF32Few<CI, CO, H, W, KH, KW, S, P, BM, TH, TWB, NIMG, LINES>> {
    using type = ConvF32Few<CI, CO, H, W, KH, KW, S, P, BM, TH, TWB, NIMG, LINES, true>;
};

}  // namespace bfuse
