// Convolution on rectangular pixel tiles: the implicit GEMM of ConvF32Lds (ops_conv_general.h: any filter size,
// stride, padding, image size and batch; channel groups of 16 under one filter tap; KS waves over the
// channel groups, each with a zero-padded LDS patch of its own; partial tiles summed in wave order) with the
// workgroup's pixels arranged as TH output rows x 16 output columns instead of 64 consecutive pixels.
//
// What that changes is the patch.  64 consecutive pixels of a wide image are part of one row, but the rows a
// wave stages are whole image rows: on a 147-wide image 4 x 149 positions for 64 outputs, of which 3 x 66 are
// read.  A TH x 16 tile needs ((TH-1) S + KH) x (15 S + KW) positions -- 6 x 18 for a 3 x 3 filter, 5.5 times
// fewer -- so the staging (global loads, scattered LDS writes) shrinks by that factor and so does the LDS a
// workgroup holds, which lets more workgroups share a CU.  The MFMA loop is ConvF32Lds's: per lane a base
// address in the patch plus a compile-time offset per tap.
//
// A patch row is a piece of an image row that starts anywhere.  It is fetched with 16-byte loads from its start on, whose floats beside the
// image are made zeros (which is what padding reads as), and is a whole number of them long in LDS, so that every float of a load has its place.  Rows past the
// image come from past the buffer's end, as zeros.  (With aligned loads each float of a vector has to find its own column and a place, if it has one: six
// vector instructions a float where this takes two.)  Output columns past
// the image (OW not a multiple of 16) and rows past it (OH not a multiple of TH) are computed on whatever the
// patch holds there and not stored.  us, before and now, with the filters through LDS (ops_conv_filters.h): 64
// channels on 56 x 56 6.6 -> 5.8.  Images of at most four channels have ConvF32Few.
//
// Replaces the same TVM-generated `conv2d` kernels of the reference as ConvF32Lds
// (scripts/configure_kernels.py:28-38,60-68); which of the two a shape gets is ConvTiling's choice.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dispatch.h"
#include "ops_conv_1x1.h"
#include "ops_conv_few.h"
#include "ops_conv_general.h"
#include "ops_conv_patch.h"
#include "ops_conv_split.h"
#include "ops_conv_tile.h"
#include "ops_gemm_split.h"
#include "ops_gemm_tile.h"
#include "wave.h"

namespace bfuse {

template <int CI_, int CO_, int H_, int W_, int KH_, int KW_, int S_, int P_, int BM_, int TH_, int KS_, int NIMG_ = 1>
struct ConvF32Rect {
    static constexpr bool MATRIX_CORES = true;   // the inner loop is a stream of MFMAs (what the fusion chooser asks)
    static constexpr int CI = CI_, CO = CO_, H = H_, W = W_, KH = KH_, KW = KW_, S = S_, P = P_, BM = BM_, TH = TH_, KS = KS_, NIMG = NIMG_;
    static constexpr int OH = (H - KH + 2 * P) / S + 1, OW = (W - KW + 2 * P) / S + 1;
    static constexpr int HW = H * W, OHW = OH * OW, T = KH * KW;
    static constexpr int CG = 16;                       // channels per group
    static constexpr int NQ = CG / 4;                   // channel quads = planes of the tile = MFMAs per tap
    static constexpr int NGROUP = CI / 16;
    static constexpr int GPW = NGROUP / KS;             // groups per wave
    static constexpr int TM = BM / 16;
    static constexpr int PB = TH;                       // 16-pixel blocks of the tile: one per output row
    static constexpr int NTX = (OW + 15) / 16, NTY = (OH + TH - 1) / TH, NPT = NTX * NTY;
    static constexpr int PR = (TH - 1) * S + KH, PC = (15 * S + KW + 3) / 4 * 4;   // patch rows / columns, whole vectors of four
    static constexpr int NPOS = PR * PC;
    // bytes of one channel quad, [position][4 channels], padded to 16 (mod 256): the planes then start one
    // 16-byte slot apart in the banks (see ops_conv.h)
    static constexpr int PLANE = (NPOS * 16 + 255) / 256 * 256 + 16;
    // The filters come to the registers through the wave's tile, before the patch is staged (ops_conv_filters.h), where they are not
    // much more than the patch: up to nine taps.
    static constexpr bool TURNED = T > 1 && T <= 9;
    using Filters = FilterRows<CI, T, BM / 16>;
    static constexpr int TILE_BYTES = TURNED && Filters::BYTES > NQ * PLANE ? Filters::BYTES : NQ * PLANE;
    static constexpr int LPC = 64 / CG;                 // lanes that share a channel while staging
    static constexpr int NVR = PC / 4;                  // vectors of a patch row
    static constexpr int NU = PR * NVR;                 // staging units (row, vector) per channel
    using Units = PatchUnits<NU, LPC>;
    using Columns = PatchColumns<W, P, 16 * S>;
    using Source = PatchSource<(long long)CG * HW>;
    static constexpr int NLD = Units::NLD;              // wave-level loads per group
    static_assert(CI % 16 == 0, "input channels: a multiple of 16");
    static_assert(CO % BM == 0 && BM % 16 == 0 && NGROUP % KS == 0, "channel tiling");
    static_assert(((KH - 1) * PC + KW - 1) * 16 + (NQ - 1) * PLANE + 16 < 65536, "tap offsets are 16-bit immediates");
    static_assert(S >= 1 && OH >= 1 && OW >= 1 && TH >= 1, "shape");

    static constexpr int NCT = CO / BM;
    static constexpr int WG_PER_IMAGE = NPT * NCT;
    static_assert(NIMG >= 1 && (long long)WG_PER_IMAGE * NIMG < (1LL << 31), "grid size");
    static constexpr Dims3 GRID{WG_PER_IMAGE * NIMG, 1, 1};
    static constexpr Dims3 BLOCK{64 * KS, 1, 1};
    static constexpr int THREADS = 64 * KS;
    static constexpr bool HAS_BARRIERS = KS > 1;
    static constexpr int PART_BYTES = KS > 1 ? KS * TM * PB * 1024 : 0;

    struct Smem {
        __attribute__((aligned(16))) unsigned char t[KS * TILE_BYTES > PART_BYTES ? KS * TILE_BYTES : PART_BYTES];
    };

    // Workgroup id -> (pixel tile, output-channel tile): id % 8 is taken as the XCD, which owns consecutive
    // pixel tiles and every channel tile of each, so that the workgroups sharing a patch use one L2.
    __device__ static __forceinline__ void tile_of(int vblock, int& pt, int& ct)
    {
        // over the pixel tiles of the WHOLE batch (image-major): with few tiles per image (an 8 x 8 image is one)
        // the channel tiles of one image would otherwise be consecutive ids, one per XCD, and each XCD would
        // fetch the image for itself (measured on the 1 x 1 layers of 8 x 8 images: 7.8 times the operands)
        constexpr int NPTB = NPT * NIMG;
        constexpr int PER_XCD = NPTB / 8;
        constexpr int FULL = 8 * PER_XCD * NCT;
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

    // accumulator layout: lane (j = column of the tile row, rg) owns output channels 4*rg+v of the block
    __device__ static __forceinline__ void store_block(float* __restrict__ Y, int co0, int oy, int ox0, int tm,
                                                       const f32x4& blk, int lane)
    {
        const int j = lane & 15, rg = lane >> 4;
        const int ox = ox0 + j;
        if (oy < OH && ox < OW) {
#pragma unroll
            for (int v = 0; v < 4; ++v) Y[(size_t)(co0 + tm * 16 + 4 * rg + v) * OHW + oy * OW + ox] = blk[v];
        }
    }

    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F,
                                               void* O, Sync sync)
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
        const int oy0 = (pt / NTX) * TH, ox0 = (pt % NTX) * 16;   // first output row / column of the tile
        const int iy0 = oy0 * S - P, ix0 = ox0 * S - P;           // image row / column of patch position (0, 0)
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int li = lane & 15, kq = lane >> 4;
        unsigned char* const tile = sm.t + wave * TILE_BYTES;

        // this lane's pixel of each block: the top-left tap of its window; channel quad kq
        const unsigned char* bbase[PB];
#pragma unroll
        for (int pb = 0; pb < PB; ++pb) bbase[pb] = tile + ((pb * S) * PC + li * S) * 16 + kq * PLANE;

        f32x4 acc[TM][PB];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) acc[tm][pb] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll 1
        for (int gi = 0; gi < GPW; ++gi) {
            const int ci0 = (wave + gi * KS) * CG;
            // A operand: Wt[co][ci0 + 4 kq + t][tap], t = 0..3: 4*T consecutive floats on a 16-byte boundary.
            f32x4 aw[TM][T];
            Filters filters;
            if constexpr (TURNED) {
                if (gi > 0) Filters::reads_done();             // of the patch before
                Filters::request(Wt, co0, ci0, 0, tile, lane);
            }
            // the filters, with BEHIND loads behind the last one's; the tile is the patch's from here on
            auto take_filters = [&](auto behind) {
                constexpr int BEHIND = decltype(behind)::value;
                if constexpr (TURNED) {
                    filters.template take<BEHIND>(0, tile, lane);
#pragma unroll
                    for (int tm = 1; tm < TM; ++tm) {
                        Filters::request(Wt, co0, ci0, tm, tile, lane);
                        filters.template take<0>(tm, tile, lane);
                    }
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                        for (int j = 0; j < T; ++j) aw[tm][j] = filters.w[tm][j];
                } else {
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) {
                        const f32x4* src = reinterpret_cast<const f32x4*>(Wt + ((size_t)(co0 + tm * 16 + li) * CI + ci0 + 4 * kq) * T);
#pragma unroll
                        for (int j = 0; j < T; ++j) aw[tm][j] = src[j];
                    }
                }
            };

            // stage the patch: LPC lanes share a channel and take the (row, vector) units of its PR patch rows in turn.  A vector of a row outside the image
            // is read past the buffer's end; floats beside the image are made zeros, which is what padding reads as (PatchColumns).
            const int cl = lane / LPC;
            int cu = lane % LPC;
            // which positions a lane stages does not change from one channel group to the next, and the compiler would
            // work out every address ahead of the loop and keep them all in registers: hidden from it
            asm volatile("" : "+v"(cu));
            const auto xr = Source::template open<(NU % LPC != 0)>(X + (size_t)ci0 * HW);
            const typename Source::Index corner = (typename Source::Index)cl * HW + iy0 * W;
            const bool inside = ix0 >= 0 && ix0 + PC <= W;          // no vector reaches beside the image
            unsigned char* const plane = tile + (cl / 4) * PLANE + (cl % 4) * 4;
            constexpr int JB = Units::JB, NBATCH = Units::NBATCH, UNROLL = (NIMG == 1 && NBATCH <= 4) ? NBATCH : 1;
            if constexpr (NBATCH > 1 || !TURNED) take_filters(std::integral_constant<int, 0>{});
#pragma unroll UNROLL
            for (int j0 = 0; j0 < NLD; j0 += JB) {
                f32x4 v[JB];
#pragma unroll
                for (int jj = 0; jj < JB; ++jj) {
                    const int u = (j0 + jj) * LPC + cu;
                    const int r = u / NVR, vi = u % NVR, iy = iy0 + r;
                    v[jj] = Source::template load<4>(xr, iy >= 0 && iy < H && u < NU ? Source::place(corner + r * W + Columns::from(ix0, vi)) : Source::outside());
                }
                if constexpr (NBATCH == 1 && TURNED) take_filters(typename Source::template Behind<JB>{});
                asm volatile("" : "+v"(cu));   // likewise: the stores work their addresses out again, one vector at a time
#pragma unroll
                for (int jj = 0; jj < JB; ++jj) {
                    const int u = (j0 + jj) * LPC + cu;
                    const int vi = u % NVR;
                    if (Units::there(j0 + jj, u)) {
                        float* const dst = reinterpret_cast<float*>(plane + u * 64);
#pragma unroll
                        for (int e = 0; e < 4; ++e) dst[4 * e] = Columns::at(v[jj], e, ix0, vi, inside);
                    }
                }
            }

            // the taps: read the next tap's operands while this one multiplies
            f32x4 b[2][PB];
#pragma unroll
            for (int pb = 0; pb < PB; ++pb) b[0][pb] = *reinterpret_cast<const f32x4*>(bbase[pb]);
#pragma unroll
            for (int tap = 0; tap < T; ++tap) {
                if (tap + 1 < T) {
                    const int noff = (((tap + 1) / KW) * PC + (tap + 1) % KW) * 16;
#pragma unroll
                    for (int pb = 0; pb < PB; ++pb) b[(tap + 1) & 1][pb] = *reinterpret_cast<const f32x4*>(bbase[pb] + noff);
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                        for (int pb = 0; pb < PB; ++pb)
                            acc[tm][pb] = __builtin_amdgcn_mfma_f32_16x16x4f32(aw[tm][(t * T + tap) / 4][(t * T + tap) % 4],
                                                                               b[tap & 1][pb][t], acc[tm][pb], 0, 0, 0);
            }
        }

        if constexpr (KS == 1) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) store_block(Y, co0, oy0 + pb, ox0, tm, acc[tm][pb], lane);
        } else {
            f32x4(*part)[TM * PB][64] = reinterpret_cast<f32x4(*)[TM * PB][64]>(sm.t);
            sync();  // the partial tiles overwrite the patches: every wave is done reading its own
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int pb = 0; pb < PB; ++pb) part[wave][tm * PB + pb][lane] = acc[tm][pb];
            sync();
            // block u is finished by wave u mod KS, summing the partials of waves 0..KS-1 in order
#pragma unroll
            for (int u0 = 0; u0 < TM * PB; u0 += KS) {
                const int u = u0 + wave;
                if (u < TM * PB) {
                    f32x4 s = part[0][u][lane];
#pragma unroll
                    for (int w = 1; w < KS; ++w) s += part[w][u][lane];
                    store_block(Y, co0, oy0 + u % PB, ox0, u / PB, s, lane);
                }
            }
        }
    }
};

// The product on the bf16 matrix cores under ConvF32Lds's name: BM output channels and 16 PB pixels of the batch for a workgroup of
// KS waves, which split the channels.  A shared tile like ConvF32Tile, whose place it takes: only what a workgroup does with it differs.
constexpr int kSplitForm = 32;
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int BM, int PB, int KS, int NIMG>
struct ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, KS, NIMG, kSplitForm> : ConvF32Tile<CI, CO, H, W, KH, KW, S, P, BM, PB % 4 == 0 ? 16 * PB : 128, 1, NIMG> {
    using Form = SwapOperands<GemmSplit<CO, CI * KH * KW, H, W, S, NIMG, BM / 16 / KS, KS, 1, 1, 16 * PB, kPix, KH, KW, P, false, (CI * KH * KW >= 256)>>;
    using Parts = typename Form::Parts;
    static constexpr int PARTS_OPERAND = Form::PARTS_OPERAND;
    static constexpr long long TILES = Form::TILES;
    static constexpr bool FITS = Form::FITS;
    static constexpr Dims3 GRID = Form::GRID, BLOCK = Form::BLOCK;
    static constexpr int THREADS = Form::THREADS, MIN_BARRIERS = Form::MIN_BARRIERS;
    using Smem = typename Form::Smem;
    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        Form::run(vblock, tid, sm, I, F, O, sync);
    }
};
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int BM, int PB, int KS, int NIMG>
struct NarrowOf<ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, KS, NIMG, kSplitForm>> {
    using type = ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, (KS > 8 && KS % 2 == 0 ? KS / 2 : KS), NIMG, kSplitForm>;
};

// The product from a patch taken apart once (ConvSplit) under that name as well: BM output channels, 32 a wave, and 16 PB pixels, TW wide
// (0: that follow each other).  (The tile it derives from says only that this is a shared tile.)
constexpr int kPatchForm = 33;
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int BM, int PB, int TW, int NIMG>
struct ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, TW, NIMG, kPatchForm> : ConvF32Tile<CI, CO, H, W, KH, KW, S, P, BM, 128, 1, NIMG> {
    using Form = SwapOperands<ConvSplit<CI, CO, H, W, KH, KW, S, P, NIMG, 2, BM / 32, 1, 16 * PB, TW>>;
    using Parts = typename Form::Parts;
    static constexpr int PARTS_OPERAND = Form::PARTS_OPERAND;
    static constexpr long long TILES = Form::TILES;
    static constexpr bool FITS = Form::FITS;
    static constexpr Dims3 GRID = Form::GRID, BLOCK = Form::BLOCK;
    static constexpr int THREADS = Form::THREADS, MIN_BARRIERS = Form::MIN_BARRIERS;
    using Smem = typename Form::Smem;
    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        Form::run(vblock, tid, sm, I, F, O, sync);
    }
};
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int BM, int PB, int TW, int NIMG>
struct SlimOf<ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, TW, NIMG, kPatchForm>> {
    using type = Slim<typename ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, TW, NIMG, kPatchForm>::Form>;
};

// The tiling the library gives a convolution it has no hand-picked one for: as many output channels per
// workgroup as keep the filter fragments of a wave within ~72 registers (the staged patch is shared by all
// of them), 64 pixels (or the whole image when it has fewer), and as many waves over the channel groups as
// leave room for two workgroups' patches in a CU's LDS.
//
// The pixels are a rectangle of 16 columns (ConvF32Rect) for filters larger than 1 x 1 on wide images whose
// rows fill their 16-column tiles well -- at least 64 outputs wide, or at least 44 (any width at a stride: 64
// consecutive outputs of a strided layer need twice the image rows) with five sixths of the tile columns in
// use -- else 64 consecutive pixels (ConvF32Lds).  Measured at batch 1024, rectangle against
// consecutive pixels: 2.3-2.5x on 147-, 149- and 299-wide images, 2.2x on 55 outputs at stride 2, 1.6x for the
// 7 x 7 on 224, 1.3x on 73 and on 48, 1.1x on 56, 54 and 44; 1.0x on 50 (14 of its 64 tile columns idle);
// 0.8-0.9x on 35- and 28-wide images and 0.45-0.55x on 17-, 8- and 7-wide ones, whose rows fill half of a
// tile or less; at stride 2 1.14x on 28 and 1.23x on 14 outputs, 0.72x on 17, 0.55x on 8, 0.41x on 7; 1 x 1
// filters have no halo to save.
//
// The rectangle has 4 rows while a wave's patch of 16 channels stays within 12.5 KB, else 2, else 1: a stride
// widens the patch (9 x 33 pixels for 4 rows of a 3 x 3 filter at stride 2, 7 x 63 for 2 rows at stride 4), and
// the smaller patch lets more workgroups share a CU and hide the staging of each other's patches: 2 rows against
// 4 at stride 2, 1.20x (112-wide, 64 channels) and 1.12x (147-wide, 32 channels); 1 row against 2 at stride 4,
// 1.4x (227-wide).
//
// A strided layer with so few output channels that it computes less per byte of image than the chip can
// (CO x taps / (2 x stride^2) flops per byte against ~20) is bound by reading the image: one workgroup then
// computes all output channels (up to 64), so that the image is read once (1.14x on the 227-wide layer).
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int NIMG>
struct ConvTiling {
    static constexpr int T = KH * KW;
    static constexpr int OH = (H - KH + 2 * P) / S + 1, OW = (W - KW + 2 * P) / S + 1;
    static constexpr int OHW = OH * OW;
    static constexpr bool RECT = T > 1 && (OW >= 64 || ((OW >= 44 || S > 1) && 6 * OW >= 5 * ((OW + 15) / 16 * 16)));
    static constexpr int patch_bytes(int th) { return ((th - 1) * S + KH) * (15 * S + KW) * 64; }
    static constexpr int TH = patch_bytes(4) <= 12800 ? 4 : patch_bytes(2) <= 12800 ? 2 : 1;
    // Images of at most four channels (ConvF32Few).  A batch writes its results 64 columns wide where three quarters of these are the image's, of filters of up to
    // 25 taps (ConvF32Few has why), on two rows; else 16 columns and eight rows of larger filters, four of smaller ones.  32 output channels a wave for up to nine
    // taps, 16 for more.  us, 256 images, 32 channels x 2 rows x 64 columns / 16 x 2 x 64 / 32 x 4 x 16: 3 x 3 on 299 at stride 2 (1024) 1065 / 1098 / 1338, on 112
    // 181 / - / 340, 5 x 5 on 149 384 / - / 371, on 299 at stride 2 779 / 690 / 763, of one channel on 112 170 / - / 244; on 150 at stride 2, 75 of 128 columns,
    // 264 / - / 229.  7 x 7 on 224 (1024), 16 channels x 8 / 7 / 4 / 12 rows and 32 x 8 / 6 / 4: 2154 / 2154 / 2206 / 2301, 2289 / 2264 / 2509.  One image,
    // 16 x 4 / 16 x 2 / 32 x 2 / 32 x 4: 5.7 / 5.9 / 5.9 / 8.0.
    static constexpr bool FEW = RECT && CI <= 4;
    static constexpr int FEW_BM = NIMG > 1 && CO % 32 == 0 && T <= 9 ? 32 : 16;
    static constexpr int few_bytes(int th, int twb) { return CI * ((th - 1) * S + KH) * ((16 * twb - 1) * S + KW) * 4; }
    static constexpr int FEW_TWB = NIMG > 1 && T <= 25 && 4 * OW >= 3 * ((OW + 63) / 64 * 64) && few_bytes(2, 4) <= 16384 ? 4 : 1;
    // Filters of many taps leave registers for fewer rows.  Eight: up to 64 registers of filters, and not where the rows of a window are many and one after the
    // other for some lane groups only (13 x 13 and 13 x 11 of one channel, 11 x 11 and 9 x 14 of two spill), or wide at stride 2, where two phases of a row are
    // kept (16 x 13 of one channel).  Four: up to 160 at a stride, 176 without.  us, four rows of ConvF32Rect as it was and now, 64 images 96 wide of four channels to 32:
    // 12 x 12 222 -> 212, 13 x 13 205 -> 204, 14 x 14 290 -> 288, 13 x 13 at stride 2 73 -> 62; of three 12 x 12 338 -> 154; of two 10 x 10 203 -> 85 (with four rows 95); of one
    // 12 x 12 250 -> 72 (76), 10 x 10 167 -> 54, 9 x 9 125 -> 39; on 224 11 x 11 at stride 4 of three to 64 427 -> 118, 12 x 12 at stride 2 of four 524 -> 483.
    using FewFilters = FilterFloats<(CI <= 4 ? CI : 4), KH, KW, 1>;
    static constexpr int FEW_NM = FewFilters::NM;
    static constexpr bool FEW_EIGHT = FEW_NM <= 64 && ((KH <= 10 && KW <= 12) || FewFilters::RPL <= 2 || KH % FewFilters::RPL == 0) && !(S == 2 && KW > 12);
    static constexpr int FEW_MOST = FEW_EIGHT ? 8 : FEW_NM <= (S == 1 ? 176 : 160) ? 4 : FEW_NM <= 200 ? 3 : 1;
    static constexpr int few_rows(int th) { return th > FEW_MOST ? FEW_MOST : th; }
    static constexpr int FEW_TH = FEW_TWB == 4 ? 2 : few_rows(NIMG > 1 && T > 25 && few_bytes(8, 1) <= 12800 ? 8 : few_bytes(4, 1) <= 25600 ? 4 : few_bytes(2, 1) <= 25600 ? 2 : 1);
    static constexpr bool FEW_LINES = FEW_TWB == 4 && OW % 16 == 0 && (long long)NIMG * CO * OHW * 4 > (1LL << 28);
    static constexpr int pick_bm()
    {
        if (CI < 16) return 16;
        if (T == 1)      // a 1x1 filter is one register per row block: as many output channels as divide CO, up to 80
            for (int bm = 80; bm > 16; bm -= 16)     // (96 measured slower than 64 on the 8x8 and 17x17 layers)
                if (CO % bm == 0) return bm;
        if (RECT && CO * T < 40 * S * S)             // bound by reading the image
            for (int bm = 64; bm > 16; bm -= 16)
                if (CO % bm == 0) return bm;
        if (CO % 64 == 0 && 4 * T <= 18) return 64;
        if (CO % 48 == 0 && 3 * T <= 18) return 48;
        if (CO % 32 == 0 && 2 * T <= 18) return 32;
        return 16;
    }
    static constexpr int BM = pick_bm();
    static constexpr int PB = OHW >= 64 ? 4 : (OHW + 15) / 16;
    static constexpr int NGROUP = CI >= 16 ? CI / 16 : 1;
    // (only the chosen form is instantiated: the other may not fit this shape at all)
    using few = ConvF32Few<CI, CO, H, W, KH, KW, S, P, FEW_BM, FEW_TH, FEW_TWB, NIMG, FEW_LINES>;
    static constexpr int TILE = std::conditional_t<FEW, few, std::conditional_t<RECT, ConvF32Rect<CI, CO, H, W, KH, KW, S, P, BM, TH, 1, NIMG>,
                                                                                ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, 1, NIMG>>>::TILE_BYTES;
    static constexpr int pick_ks()
    {
        // a rectangle gets no more waves than it has rows: the sum of the waves' partial tiles costs the same
        // whatever the rows' arithmetic (4 waves on 2 rows: 0.92x of 2 waves on the 112-wide stride-2 layer)
        const int most = RECT ? TH : 4;
        if (most >= 4 && NGROUP % 4 == 0 && 4 * TILE <= 80 * 1024) return 4;
        if (most >= 2 && NGROUP % 2 == 0 && 2 * TILE <= 80 * 1024) return 2;
        return 1;
    }
    static constexpr int KS = pick_ks();
    // A 1 x 1 filter on enough pixels to give every SIMD of the chip a 64-pixel tile is streamed (Conv1x1F32:
    // no LDS patch, no partial sums), with as many output channels per workgroup as divide CO, up to 80.
    // Measured at batch 1024 against the staged form: 2.1x on 64 -> 64 channels at 56 x 56 (5.2 TB/s of image and
    // output), 1.3-1.7x on the 35 x 35 layers, 1.8x on 73 x 73, 1.2-1.3x on 17 x 17 and 8 x 8 with 768-2048 channels
    // (120 TFLOP/s), 1.7x on 256 -> 256 at 56 x 56 (117 TFLOP/s).
    static constexpr bool STREAM = T == 1 && P == 0 && CI % 16 == 0 && CO % 16 == 0 && (long long)((OHW + 63) / 64) * NIMG >= 1024;
    static constexpr int stream_bm()
    {
        for (int bm = 80; bm > 16; bm -= 16)
            if (CO % bm == 0) return bm;
        return 16;
    }
    using staged = std::conditional_t<FEW, few, std::conditional_t<RECT, ConvF32Rect<CI, CO, H, W, KH, KW, S, P, BM, TH, KS, NIMG>,
                                                                   ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, KS, NIMG>>>;
    // Those that write most, one wave with a patch of a few KB, are held to eight workgroups per CU, so that fewer rows of results are written at a time
    // (LdsReserve): 3 x 3 on 299 x 299 at stride 2 1065 -> 985 us, with six 1112; of 5 x 5 filters 714 -> 798.
    static constexpr int RESERVE = FEW && FEW_TWB == 4 && T <= 9 && (int)sizeof(typename staged::Smem) < 163840 / 8 - 1024
                                       ? 163840 / 8 - (int)sizeof(typename staged::Smem) : 0;
    using held = std::conditional_t<(RESERVE > 0), LdsReserve<staged, (RESERVE > 0 ? RESERVE : 1)>, staged>;
    // A batch with enough pixels for two workgroups per CU goes to the shared-tile form, with the largest tile whose
    // part of each wave is at least twelve 16 x 16 blocks: measured at batch 1024 over the 3 x 3 and 5 x 5 layers it
    // takes 0.39-0.80 of the time of the per-wave forms above (108-146 TFLOP/s against 52-118); with eight blocks per wave
    // (32 x 64) 1.04-1.08 at stride 1.  96 channels before 128: 141 against 139 TFLOP/s on 288 -> 384; 64 x 256 pixels, one
    // wave over the channels, against 64 x 128, two: 136 against 88 on 64 -> 64 at 56 x 56.
    static constexpr int tile_bm() { return CO % 96 == 0 ? 96 : CO % 128 == 0 ? 128 : CO % 160 == 0 ? 160 : CO % 64 == 0 ? 64 : CO % 48 == 0 ? 48 : CO % 80 == 0 ? 80 : CO % 32 == 0 ? 32 : 16; }
    // At stride 1 half the channels and twice the pixels: the patch of 256 consecutive pixels of a row or image has few more
    // rows than that of 128, the workgroup takes 32-38 KB of LDS instead of 42-48, and more of them share a CU (1.00-1.01x
    // on six layers: 137 against 136 TFLOP/s for 256 -> 256 on 14 x 14, 137.4 against 137.2 for 96 -> 96 on 35 x 35).  Not at
    // stride 2, whose patch is four times the pixels (0.95-1.00x), nor on images so small that 256 pixels are several of
    // them (8 x 8: 0.99x).
    static constexpr bool HALF = S == 1 && tile_bm() >= 96 && OHW >= 128;
    static constexpr int TBM = HALF ? tile_bm() / 2 : tile_bm(), TWM = TBM >= 96 ? 2 : 1, TPB0 = TBM >= 96 ? 8 : TBM >= 48 ? 16 : 32;
    // A quarter more pixels per tile where that leaves less of the last round idle.  A CU multiplies two workgroups' tiles in
    // the time of two, so a round is 256 tiles: 512 -> 512 channels on 7 x 7 is 6.13 rounds (7) of 128 pixels but 4.9 (5) of
    // 160: 137 against 126 TFLOP/s; 256 -> 256 on 14 x 14 138 against 137; 256 -> 512 on 14 x 14 at stride 2 131 against 119.
    // A gain of two in a hundred by this count was 0.99-1.01x.  At most twenty blocks per wave: they take 160 registers.
    static constexpr double filled(int pb)
    {
        const long long tiles = ((long long)OHW * NIMG + 16 * pb - 1) / (16 * pb) * (CO / TBM);
        return (double)OHW * NIMG * (CO / TBM) / (16 * pb) / 256 / (double)((tiles + 255) / 256);
    }
    static constexpr bool tiled(int pb)
    {
        if constexpr (T > 1 && CI >= 16 && CI % 4 == 0 && KH >= S && TBM >= 32 && (long long)OHW * NIMG >= 512LL * 16 * TPB0 * TBM / CO)
            return pb == TPB0 ? ConvF32Lds<CI, CO, H, W, KH, KW, S, P, TBM, TPB0, 4, NIMG, TWM>::FITS
                              : TBM / 16 * (TPB0 / 4 * 5) <= 80 && ConvF32Lds<CI, CO, H, W, KH, KW, S, P, TBM, TPB0 / 4 * 5, 4, NIMG, TWM>::FITS;
        return false;
    }
    static constexpr int TPB = filled(TPB0 / 4 * 5) > 1.03 * filled(TPB0) && tiled(TPB0 / 4 * 5) ? TPB0 / 4 * 5 : TPB0;
    // 1 x 1 filters likewise, as a matrix product (GemmTile): 1.01-1.19x of the streamed form at stride 1 (119-145 TFLOP/s on the
    // layers of 768 and more channels, 4.0-5.1 TB/s on those of few), 1.4-1.9x at stride 2, where that one reads element
    // by element.  Three buffers of 16 channels for 128-pixel tiles (134 against 124 TFLOP/s with two of 32 on 768 -> 192),
    // two for 256-pixel ones, which are bound by memory and want more workgroups per CU.
    static constexpr int GBM = CO % 96 != 0 && CO % 224 == 0 ? 224 : tile_bm(), GWM = GBM >= 96 ? 2 : 1, GBN = GBM >= 96 ? 128 : 256;
    // Only where the streamed form would do, which also keeps one sum over all channels.
    using product = GemmTile<CO, CI, H, W, S, NIMG, GBM, GBN, GWM, 16, kPix, GWM == 2 ? 3 : 2>;
    static constexpr bool is_product()
    {
        if constexpr (STREAM && tile_bm() >= 32 && (long long)((OHW + 3) / 4 * 4) * NIMG / GBN * (CO / GBM) >= 512) return product::FITS;
        return false;
    }
    // Filters larger than 1 x 1: as a product on the bf16 matrix cores whose second operand is gathered from the images (GemmSplit),
    // on at least two rounds of tiles over the CUs.  The tile is the largest of 256 x 128 (eight waves), 128 x 128, 192 x 64 (four
    // waves, two workgroups a CU), 160 x 128 (ten waves of 16 rows), 96 x 64 (two waves) and 64 x 128 (four of 16 rows) whose rows
    // divide the channels.  (Those at stride 1 have since gone on to the patch above, except channels that are no groups of 32.)  Batch 1024, us, shared tiles before
    // (all on one card; others hold 0.93-1.00 of the clock): 256 -> 256 on 14 x 14 1712 -> 1033 (128 x 128: 1.09x that), 512 on 7 x 7
    // 1720 -> 1136, 128 on 28 x 28 1692 -> 1122, 448 -> 384 on 8 x 8 1381 -> 882 (192 x 64: 1.08x), 288 -> 384 at stride 2 4153 -> 2838
    // (192 x 128 and x 64: 1.10x), 80 -> 192 on 73 x 73 10209 -> 7393, 192 -> 320 at stride 2 521 -> 378 (128 x 128 on 2.5 tiles: 433; five
    // waves of 32 rows twice 477).  Few channels
    // give the gathered operand few uses for what taking it apart costs: 96 -> 96 on 35 x 35 1506 -> 1169 (96 x 128 on four waves 1.01x,
    // on six of 16 rows 1.3x), 64 -> 96 1056 -> 852, 64 -> 64 on 56 x 56 1740 -> 1504 (64 x 64 1.02x, 64 rows a wave 1.2x), 5 x 5 48 -> 64
    // 1432 -> 1161, 32 -> 64 on 147 x 147 6802 -> 5938, 16 -> 64 at stride 4 1338 -> 865; but at stride 2, where a load of the gather
    // touches twice the lines and the tile's patch was loaded once, 32 -> 64 on 147 x 147 1864 -> 1891.
    static constexpr int SBM = CO % 256 == 0 ? 256 : CO % 128 == 0 ? 128 : CO % 192 == 0 ? 192 : CO % 160 == 0 ? 160 : CO % 96 == 0 ? 96 : 64;
    // 256 rows on 112 pixels instead of 128 where that leaves less of the last round over the CUs idle: 256 -> 512 on 14 x 14 at stride 2 is 3.25 rounds (4) of
    // 128 but 3.7 of 112, 611 -> 585 us; 128 -> 256 on 28 x 28 573 -> 568.
    static constexpr int ROUNDS8 = (int)(((long long)((OHW + 3) / 4 * 4) * NIMG + 127) / 128 * (CO / 256) + 255) / 256, ROUNDS7 = (int)(((long long)((OHW + 3) / 4 * 4) * NIMG + 111) / 112 * (CO / 256) + 255) / 256;
    static constexpr int PB256 = 112 * ROUNDS7 < 0.97 * 128 * ROUNDS8 ? 7 : 8;
    using split = ConvF32Lds<CI, CO, H, W, KH, KW, S, P, SBM, SBM == 256 ? PB256 : SBM == 192 || SBM == 96 ? 4 : 8, SBM == 256 ? 8 : SBM == 160 ? 10 : SBM == 96 ? 2 : 4, NIMG, kSplitForm>;
    // Filters of 31 and more taps are left to the per-wave forms: 7 x 7 on RGB takes 2154 us there and took 2363 as a product, a window with one element that is
    // not zero came out up to 2.4 u off instead of 1 as a product, and one wave without barriers can be thread-fused with any operator.
    static constexpr bool is_split()
    {
        // (the table of taps is made at compile time)
        if constexpr (T > 1 && T < 31 && CI % 16 == 0 && CI * T <= 32768 && CO % SBM == 0 && !(SBM == 64 && S == 2))
            return split::FITS && split::TILES >= 512;
        return false;
    }
    // 3 x 3 filters at stride 1 on whole groups of 32 channels take the images apart once for all taps (ConvSplit, which has the figures: 0.71-0.92 of
    // split's time on eleven layers, 0.75-0.89 on ten others from 14 x 14 to 14 x 300), where a tile of the most output channels up to 128 that divide theirs fits twice
    // into a CU's LDS with at most 15 % of it (tiles of 128 channels: 17) outside the images: of 128, 112 or 96 consecutive pixels, 28 x 4, 16 x 7 and 12 x 12, the one that
    // computes least besides.  Measured: 14 x 14 on 112 900 us, on 96 926; 7 x 7 on 96 972, on 112 (one tile a CU) 1062; 8 x 8 on 128 755, on 64 793; 35 x 35 on 12 x 12
    // 702, on 12 x 8 760, on 36 x 4 806; 56 x 56 on 28 x 4 1242, on 16 x 8 1372; 147 x 147 on 16 x 7 4338, on 12 x 12 4424; 26 x 26
    // on 28 x 4 (16 % outside) 1728, split 1785.  (There 224 consecutive pixels on eight waves, one tile a CU, take 1618, but beside their 150 KB of LDS a
    // thread-fused partner has 13 KB, and a block-fused one runs only on CUs without such a tile.)
    // Tiles have at least 64 of the output channels: a row tile takes its patch apart for itself, and 32 -> 32 on 149 x 149 was on the fp32
    // instructions before, where a window with one element that is not zero is at most 1 u off and here up to 2.4 (2975 instead of 3479 us).
    static constexpr int QBM = CO % 128 == 0 ? 128 : CO % 96 == 0 ? 96 : 64;
    template <int PB, int TW> using patch = ConvF32Lds<CI, CO, H, W, KH, KW, S, P, QBM, PB, TW, NIMG, kPatchForm>;
    // what a tile costs a pixel: those outside the image, and a sixteenth part of a wave's columns that every tile takes besides
    template <int PB, int TW>
    static constexpr double patch_cost()
    {
        using F = patch<PB, TW>;
        if constexpr (F::FITS && (PB != 9 || CI <= 128)) {   // (nine blocks of columns take all registers there are)
            const double pixels = 16.0 * PB * (double)F::TILES / (CO / QBM) / ((double)OHW * NIMG);
            if (2 * (int)sizeof(typename F::Smem) <= 163840 && pixels <= (QBM == 128 ? 1.17 : 1.15)) return pixels * (1 + 1.0 / PB);
        }
        return 1e9;
    }
    static constexpr int patch_form()     // 100 TW + PB, or 0
    {
        if constexpr (KH == 3 && KW == 3 && S == 1 && CI % 32 == 0 && CO % QBM == 0 && CI * T <= 32768 && (long long)OHW * NIMG >= 512LL * 128 * QBM / CO) {
            const int f[] = {8, 7, 6, 2807, 1607, 1209};
            const double c[] = {patch_cost<8, 0>(), patch_cost<7, 0>(), patch_cost<6, 0>(), patch_cost<7, 28>(), patch_cost<7, 16>(), patch_cost<9, 12>()};
            return least(f, c);
        }
        return 0;
    }
    template <int N>
    static constexpr int least(const int (&f)[N], const double (&c)[N])
    {
        int best = 0;
        for (int i = 1; i < N; ++i)
            if (c[i] < c[best]) best = i;
        return c[best] < 1e8 ? f[best] : 0;
    }
    // 1 x 1 filters on 256 and more channels likewise, also on 224 x 128 tiles (seven waves).  us, GemmTile before (the filters taken apart by every workgroup; GemmSplit has what it gave to do that once): 768 -> 192 on
    // 17 x 17 641 -> 525 (twelve waves of 16 rows 0.96x that, but no register is left beside twelve waves), 160 573 -> 447, 128 455 -> 344,
    // 1280 -> 448 on 8 x 8 521 -> 378, 384 450 -> 314, 320 377 -> 292, 192 233 -> 179, 2048 -> 448 824 -> 582, 256 -> 256 on 56 x 56
    // 3034 -> 2502, 256 -> 512 at stride 2 145 -> 121.  (160 rows are ten waves on four SIMDs, bound by their LDS reads: 155 TFLOP/s where 256 x
    // 128 tiles have 207; five waves of 32 rows, 64 or 160 pixels, and lean ones are slower.)  On fewer channels the tile's ends are too much of it: 128 -> 256 at stride 2
    // 152 against 177, 64 -> 128 202 against 218; 64 output channels 394 against 383-410.
    static constexpr int S1BM = CO % 256 == 0 ? 256 : CO % 128 == 0 ? 128 : CO % 224 == 0 ? 224 : CO % 192 == 0 ? 192 : 160;
    static constexpr int S1WR = S1BM == 256 ? 8 : S1BM == 224 ? 7 : S1BM == 160 ? 10 : 4;
    using split_product = GemmSplit<CO, CI, H, W, S, NIMG, S1BM / 16 / S1WR, S1WR, 1, 1, S1BM == 256 ? 16 * PB256 : S1BM == 192 ? 64 : 128, kPix, 1, 1, 0, false, true>;
    static constexpr bool is_split_product()
    {
        if constexpr (STREAM && CI >= 256 && CO % S1BM == 0) return split_product::FITS && split_product::TILES >= 512;
        return false;
    }
    template <int FORM, class Else> struct pick { using type = Else; };
    template <class Else> struct pick<3, Else> { using type = split; };
    template <class Else> struct pick<5, Else> { using type = patch<patch_form() % 100, patch_form() / 100>; };
    template <class Else> struct pick<4, Else> { using type = SwapOperands<split_product>; };
    template <class Else> struct pick<1, Else> { using type = ConvF32Lds<CI, CO, H, W, KH, KW, S, P, TBM, TPB, 4, NIMG, TWM>; };
    template <class Else> struct pick<2, Else> { using type = SwapOperands<product>; };
    using type = typename pick<(patch_form() > 0) ? 5 : is_split() ? 3 : is_split_product() ? 4 : is_product() ? 2 : tiled(TPB) ? 1 : 0, std::conditional_t<STREAM, Conv1x1F32<CI, CO, H, W, S, stream_bm(), 4, NIMG>, held>>::type;
};
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int NIMG = 1>
using ConvF32Auto = typename ConvTiling<CI, CO, H, W, KH, KW, S, P, NIMG>::type;

}  // namespace bfuse
