// fp32 matrix product on the bf16 matrix cores: every operand as the sum of three bf16 (split.h), six MFMAs of 16 times the
// fp32 rate for each of the fp32 ones they replace.
//
//   C[m][n] = sum_k A[m][k] * B(k, n)
//
// The fp32 forms (GemmF32Dma, GemmTile) run at 143 - 150 TFLOP/s on large products, the rate of the fp32 matrix instructions.
// Six bf16 products at the 1.74 - 2.07 PFLOP/s that random operands leave the chip are 290 - 345 of these.  What stands in between is
// taking the operands apart: six vector instructions an element, of which two go between two MFMAs of a wave almost for free
// (17 -> 19 clocks) and more do not.  So the tile is as large as it can be (an element of A is used BN times, one of B BM times)
// and every element is taken apart once in the workgroup:
//   * a wave owns 16 TM rows of A alone and takes them apart in its registers: lane (i, q) loads A[i][8q .. 8q + 7], which is
//     the MFMA's operand;
//   * B is shared: a thread takes eight k of a column apart and writes them to LDS, [part][8-k octet][column][16 bytes], where
//     the fragment reads of a wave are 256 consecutive bytes for each of its four octets: no bank is met twice.  kRows, where four lanes have
//     a column's octets: column c of octet o at c ^ 4 o, so that the writes do not meet a bank four times either (TURNED; 512 x 512 x 128 of 32 heads 18.9 -> 18.6 us, 512 x 128 x 512
//     18.3 -> 17.9, 1024 products 0.98-0.99x; reductions of 64, two stages, 1.01x: not these);
//   * three LDS buffers and one barrier per stage of 32 k.  While stage s is multiplied, the stage two ahead is taken apart and
//     written and the A of the next one taken apart, dealt between the MFMAs; the loads are a stage ahead of that;
//   * PREP: A is taken apart by a kernel that runs before this one (SplitParts), once instead of by every workgroup that has its rows. A
//     wave's three loads for 16 rows and 32 k go straight into the registers that it multiplies from, a stage ahead; that they are 1.5 times the bytes is what it
//     costs. Filters, and activations that many column tiles share. us, in turn on one card: 768 -> 192 on 17 x 17 531 -> 472, -> 160 461 -> 447, -> 128 352 ->
//     340, 1280 -> 384 on 8 x 8 321 -> 309, 2048 -> 192 283 -> 260, 80 -> 192 of 3 x 3 on 73 x 73 7520 -> 6700, 64 -> 192 at stride 2 4186 -> 3650, 288 -> 384 2890 -> 2750, 192 -> 320 382 ->
//     372, 1024 x 4096 x 14336 (on 112 columns, 512 tiles for 448) 520 -> 505, 512 x 4096 x 4096 94 -> 91: 0.945 in the geometric mean of 26 operators, the same bits.  The
//     rows' kernel is 5 us for filters and 8 for 1024 x 4096, with its launch 3 more: 1024 x 4096 x 4096 170 -> 173, 1024 x 14336 x 4096 571 -> 574, 1024 x 768 x 3072 33 -> 38, and 16 -> 64 channels (K = 144) 1.01x stay without;
//   * products with few tiles give two groups of waves the even and the odd stages (KG = 2): two waves per SIMD hide each
//     other's waits, and the groups' sums meet in LDS at the end.
// The operands of an MFMA are given in the order (B, A), so that a lane ends up with four consecutive columns of a row.
//
// What rounds the sum is one addition per partial sum of four stages (`part`; two where there are 9 - 20 of them), of which each
// stage's MFMAs round only the small beginning: 2-norm errors against 64 bits are below those of the fp32 forms at every operator, the
// largest error over the result's root mean square, given second here, at all but 64 -> 128 channels on 56 x 56 (1.28e-6 and 1.36e-6).  Reduction of 14336 2.2e-7, 1.1e-6 (GemmF32Dma 1.1e-6, 6.6e-6), 4096 1.9e-7, 1.5e-6 (5.8e-7,
// 4.2e-6), 768 1.6e-7, 9.4e-7 (2.5e-7, 1.5e-6), 128 1.5e-7, 2.8e-6 (GemmTile 2.0e-7, 3.2e-6), 64 9.3e-8, 1.5e-6 (1.4e-7, 2.3e-6); 3 x 3
// filters on 576 1.1e-7, 8.6e-7 (ConvF32Tile 1.4e-7, 1.0e-6; with four stages 1.5e-7, 1.2e-6), on 1152 1.7e-7, 1.1e-6 (1.9e-7, 1.5e-6).
// (The five small products summed apart from the large one instead, two sets of registers as well, leave one addition per stage:
// 1.0e-7 but 1.5e-6 on 576, 4.0e-7, 4.6e-6 on 4096; 1-3 % faster on large tiles, where the sums' additions take the place of other
// vector work.)  What three bf16 cannot hold is multiplied again with the fp32 MFMAs (see split.h): a wave whose results are not
// all finite, and the workgroup if a thread has met a value that is more than its parts (the ors
// that notice it take 0.2 % of the time in the mean, 2 % of 512 and 1024 x 4096 x 4096).  That pass is bound by the fp32 MFMAs and
// by loads that waves do not share; a tile takes 1.5 - 4 times what it took (us, no such value / one / one in every row of A;
// in brackets with four dependent k at a time): 1024 x 4096 x 14336 655 / 1630 (7923) / 1740, 1024 x 4096 x 4096 171 / 463 (2573) /
// 500, 512 x 512 x 128 of 32 heads 20 / 44 (185) / 49, 256 -> 256 on 14 x 14 1285 / 1282 (2957) / 4290 (18392), all on
// uniform operands and a card that had been idle.
//
// Reductions of up to four stages are one partial sum: no second set of accumulators, every stage compiled apart, and so nothing
// loaded or taken apart past the last one (with two stages that was half of it): 512 x 128 x 512 545 -> 499 us.
//
// Measured (us, before = GemmF32Dma; uniform operands, two cards): 1024 x 4096 x 14336 828 -> 508-547 (220-237 TFLOP/s), 1024 x 14336 x
// 4096 812 -> 539-569, 1024 x 4096 x 4096 236 -> 155-166, 512 x 4096 x 14336 460 -> 253-270, 512 x 4096 x 4096 118 -> 90-97, 1024 x 768 x
// 3072 38 -> 30-31.  Smaller tiles than 64 x 64 a workgroup take more time than the fp32 forms: 1024 x 3072 x 768 63 (64 x 96
// tiles) against 39.
//
// B comes in one of two layouts, as in GemmTile: kPix, planes of n for each k ([K, N] is one image of N pixels); kRows, rows
// contiguous along k, NIMG independent products.  With a filter of KH x KW taps (kPix) the product is a convolution: A holds the
// filters as they lie in memory, k counts (channel, tap), and what a column loads for k is its window's element.  All lanes of a
// load want the same k, so where the element lies from the window's first one comes from a table by a scalar load; padding is a
// lane whose bit for that tap is set and which therefore reads past the buffer (two vector instructions a load).  Every element
// is taken apart once for each tap it is under: 256 -> 256 channels on 14 x 14, batch 1024, 1715 -> 1047-1104 us (214-226 TFLOP/s; 3 x 3 filters
// at stride 1 do without that in ConvSplit, 901 us); ConvTiling has the other layers and where the line to the shared tiles lies.  A row tile (kRows: also a column tile) that does not
// divide the problem starts a tile before its end and leaves its neighbour's results to it: one of the two may be done again.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "dispatch.h"
#include "ops_gemm_tile.h"
#include "split.h"
#include "wave.h"

namespace bfuse {

// The parts of a matrix [M, K] of fp32, as a kernel of its own leaves them in a workspace (Prepares, fuse.h) for one that multiplies it: for
// every 16 rows and 32 k (a stage) the three parts one after the other, each as the MFMA's operand, 16 bytes a lane.  In front of them: where the matrix
// itself lies, and a word for every 16 rows and eight stages that is not zero if a value is more than its parts.  TAPS > 1: k counts (channel, tap), and
// taps are put behind the channels, 32 of which are a stage's k then, stage (channels, tap) (ConvSplit); a word for every 32 channels.
// One wave takes a stage apart at a time; a lane's values are TAPS apart, so a wave's loads touch 16 rows, of which the other taps' then
// come from the caches: 256 x 2304 in 5 us.
template <int M, int K, int TAPS, bool ON = true>
struct SplitParts {
    static_assert(!ON || (M % 16 == 0 && K % 8 == 0 && (TAPS == 1 || K % (32 * TAPS) == 0)), "parts");
    static constexpr int PARTS_THREADS = 256;
    static constexpr int STAGES = (K + 31) / 32, CHUNK = TAPS > 1 ? TAPS : 8, CHUNKS = (STAGES + CHUNK - 1) / CHUNK;
    static constexpr int BLOCK_BYTES = STAGES * 3072, HEAD = (64 + M / 16 * CHUNKS * 4 + 1023) / 1024 * 1024;
    static constexpr unsigned PARTS_GRID = M / 16 * CHUNKS;
    static constexpr size_t PARTS_BYTES = (size_t)HEAD + (size_t)(M / 16) * BLOCK_BYTES;

    __device__ static __forceinline__ const void* source(const void* parts) { return *static_cast<const void* const*>(parts); }
    __device__ static __forceinline__ const unsigned char* block(const void* parts, int b) { return static_cast<const unsigned char*>(parts) + HEAD + (size_t)b * BLOCK_BYTES; }
    // Whether a value of 16-row blocks b .. b + n - 1 is more than its parts, some lane's share of that.
    __device__ static __forceinline__ unsigned inexact(const void* parts, int b, int n, int lane)
    {
        const unsigned* const words = reinterpret_cast<const unsigned*>(static_cast<const unsigned char*>(parts) + 64) + b * CHUNKS;
        unsigned any = 0;
        for (int i = lane; i < n * CHUNKS; i += 64) any |= words[i];
        return any;
    }
    __device__ static __forceinline__ void take_apart(const void* operand, void* parts)
    {
        const int b = blockIdx.x / CHUNKS, chunk = blockIdx.x % CHUNKS, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
        const float* const row = static_cast<const float*>(operand) + (size_t)(16 * b + (lane & 15)) * K;
        __shared__ unsigned more;
        if (threadIdx.x == 0) more = 0;
        if (blockIdx.x == 0 && threadIdx.x == 0) *static_cast<const void**>(parts) = operand;
        __syncthreads();
        unsigned left = 0;
        for (int s = chunk * CHUNK + wave; s < (chunk + 1) * CHUNK && s < STAGES; s += PARTS_THREADS / 64) {
            float x[8];
            const int k = TAPS > 1 ? (chunk * 32 + (lane >> 4) * 8) * TAPS + s % TAPS : s * 32 + (lane >> 4) * 8;
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = K % 32 == 0 || k < K ? row[k + e * TAPS] : 0.f;
            unsigned p[3][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) split2(x[2 * j], x[2 * j + 1], p[0][j], p[1][j], p[2][j], left);
            unsigned char* const to = static_cast<unsigned char*>(parts) + HEAD + (size_t)b * BLOCK_BYTES + (size_t)s * 3072 + lane * 16;
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(to + q * 1024) = u32x4{p[q][0], p[q][1], p[q][2], p[q][3]};
        }
        if (split_inexact(left)) more = 1;
        __syncthreads();
        if (threadIdx.x == 0) reinterpret_cast<unsigned*>(static_cast<unsigned char*>(parts) + 64)[b * CHUNKS + chunk] = more;
    }
};

// M, K, H, W, S, NIMG, LAYOUT: as in GemmTile.  TM 16-row blocks of a wave, WR waves over the rows and WN over the BN columns, KG
// groups of such waves over the stages.  LEAN: one set of A's parts, taken apart at the top of the stage, instead of the next one's
// beside this one's: 12 TM registers less for a stage that begins without MFMAs, which other workgroups of the CU fill.  PREP: I is A's parts.
// LINES_: whether results are written a line at a time and past the caches (-1: by their size).
template <int M_, int K_, int H_, int W_, int S_, int NIMG_, int TM_, int WR_, int WN_, int KG_, int BN_, int LAYOUT_, int KH_ = 1, int KW_ = 1, int P_ = 0,
          bool LEAN_ = (LAYOUT_ == kRows && K_ <= 256), bool PREP_ = false, int LINES_ = -1>
struct GemmSplit {
    using Parts = SplitParts<M_, K_, 1, PREP_>;
    static constexpr int PARTS_OPERAND = PREP_ ? 0 : -1;
    static constexpr bool MATRIX_CORES = true;   // the inner loop is a stream of MFMAs (what the fusion chooser asks)
    static constexpr int M = M_, K = K_, H = H_, W = W_, S = S_, NIMG = NIMG_, TM = TM_, WR = WR_, WN = WN_, KG = KG_, BN = BN_, LAYOUT = LAYOUT_, KH = KH_, KW = KW_, P = P_;
    static constexpr int T = KH * KW, CI = K / T;                                // kPix: taps, channels of the images
    static constexpr bool LEAN = LEAN_, PREP = PREP_;
    static_assert(!PREP || !LEAN, "lean: one set of A's parts");
    static constexpr int NWAVE = WR * WN * KG, THREADS = 64 * NWAVE, GT = 64 * WR * WN, BM = 16 * TM * WR, TN = BN / WN / 16;
    static constexpr int NS = (K + 31) / 32, NIT = NS / KG, TAIL = K % 32;       // stages, those of a group, k of the last one if not 32
    static constexpr int OH = (H - KH + 2 * P) / S + 1, OW = (W - KW + 2 * P) / S + 1, HW = H * W, OHW = OH * OW;
    static constexpr int OHWP = (OHW + 3) / 4 * 4;                               // columns of an image, whole chunks of four
    static constexpr int MT = (M + BM - 1) / BM;
    static constexpr int NT = LAYOUT == kRows ? (W + BN - 1) / BN : (int)(((long long)OHWP * NIMG + BN - 1) / BN);
    static constexpr int NIMAGES = LAYOUT == kRows ? 1 : (BN + OHWP - 2) / OHWP + 1;   // images a tile can touch
    // Columns of an octet as the units (a column's eight k) are dealt to the threads: whole waves of them for filters larger than
    // 1 x 1, a wave's units being one octet's.
    static constexpr int BU = T > 1 ? (BN + 63) / 64 * 64 : BN;
    static constexpr int NUJ = (4 * BU + GT - 1) / GT;                           // units of a thread and stage
    // a thread's units lie the same way apart for all threads (kRows: GT / 4 columns, kPix: GT / BU octets of one column), so that
    // one address serves them all
    static constexpr bool EVEN = 4 * BU % GT == 0 && GT % (LAYOUT == kRows ? 4 : BU) == 0;
    static constexpr int NUB = EVEN ? 1 : NUJ;
    static_assert(BN % (16 * WN) == 0 && K % 8 == 0 && NS % KG == 0 && M >= BM && (LAYOUT == kPix || (W >= BN && H == 1 && S == 1)), "tile");
    // 31-bit offsets; padding is read through one that lies past the buffer
    static constexpr bool FITS = (long long)BM * (PREP ? NS * 32 * 6 : K * 4) < (1LL << 31) && (long long)(NIMAGES < NIMG ? NIMAGES : NIMG) * CI * HW * 4 < (1LL << (T == 1 ? 31 : 29));
    static constexpr bool TURNED = LAYOUT == kRows && NS > 2;
    static constexpr int PLANE = 4 * BN * 16, BUF = 3 * PLANE, NBUF = NIT < 3 ? NIT : 3;
    static constexpr int SUMMED = NIT > 8 && NIT <= 20 ? 2 : 4;                     // stages of a partial sum (error and time: above)
    static constexpr int TILES = MT * NT;
    static constexpr Dims3 GRID{LAYOUT == kRows ? TILES * NIMG : TILES, 1, 1};
    static constexpr Dims3 BLOCK{THREADS, 1, 1};
    static constexpr bool HAS_BARRIERS = true;
    static constexpr bool LOOP_BARRIERS = true;
    static constexpr int MIN_BARRIERS = NIT;
    static constexpr int RED_BYTES = (KG - 1) * BM * BN * 4;                     // partial sums of the groups
    // Results that are more than the last-level cache holds (256 MB) and lie in whole lines (two blocks of columns): every line is written at once and past the
    // caches.  Otherwise a store is 64 bytes of sixteen rows, and the results take the place of everything else in the caches.  us, launched again and again / in turn
    // with a layer of 900 MB: 1024 products 512 x 64 x 512 296 -> 256 / 295 -> 281, 1024 x 64 x 512 588 -> 565 / 587 -> 568, 512 x 128 x 512 453 -> 450 / 459 -> 451,
    // 256 -> 256 channels on 56 x 56 2438 -> 2377 / 2436 -> 2374.  Not 256 MB themselves: 256 x 80 x 256 105 -> 86 / 99.5 -> 100.2, 256 x 64 x 256 83 -> 68 / 76.7 -> 77.3,
    // where the gain is that operands of 134 - 168 MB stay in the last-level cache for the next launch over the same ones.  Whole lines through the caches gain 0-1 %,
    // 64 bytes past them lose up to 5 % (512 x 128 x 512).  Smaller results stay in that cache for what reads them (256 x 256 x 64, 67 MB, launched again and again
    // would take 75 us for 81).
    static constexpr bool IN_LINES = TN % 2 == 0 && M % BM == 0 && (LAYOUT == kRows ? W % BN == 0 && W % 32 == 0 : OHW % 32 == 0);
    static constexpr bool LINES = IN_LINES && (LINES_ >= 0 ? LINES_ > 0 : (long long)NIMG * M * (LAYOUT == kRows ? W : OHW) * 4 > (1LL << 28));
    static_assert(LINES_ <= 0 || LINES, "whole lines");

    struct Smem {
        __attribute__((aligned(16))) unsigned char t[NBUF * KG * BUF > RED_BYTES ? NBUF * KG * BUF : RED_BYTES];
        unsigned inexact;
    };

    // Filters larger than 1 x 1: where element k = (channel, row, column) of a window lies from its first one, in bytes, times
    // eight, and the tap's number in the low five bits; past the last k a tap that no window has.
    struct Taps {
        unsigned at[T > 1 ? NS * 32 : 1];
        constexpr Taps() : at{}
        {
            for (int k = 0; T > 1 && k < NS * 32; ++k) at[k] = k < K ? (unsigned)((k / T * HW + k % T / KW * W + k % KW) * 4) << 3 | (unsigned)(k % T) : 31u;
        }
    };
    __device__ static constexpr Taps TAPS{};
    static_assert(T == 1 || (LAYOUT == kPix && BN >= 64 && T < 31 && K % T == 0), "taps");

    // (column tile, row tile), dealt so that the row tiles of one column tile follow each other on one XCD
    template <int NT = GemmSplit::NT>
    __device__ static __forceinline__ void tile_of(int vblock, int& nt, int& mt)
    {
        constexpr int PER_XCD = NT / 8;
        constexpr int FULL = 8 * PER_XCD * MT;
        if (vblock < FULL) {
            const int xcd = vblock & 7, slot = vblock >> 3;
            nt = xcd * PER_XCD + slot / MT;
            mt = slot % MT;
        } else {
            const int rem = vblock - FULL;
            nt = 8 * PER_XCD + rem / MT;
            mt = rem % MT;
        }
    }

    static constexpr unsigned B_K = LAYOUT == kRows ? 4 : HW * 4;                   // bytes from one k of a column to the next
    // Offset of B(0, column c of the tile); past the buffer if there is none.  Filters larger than 1 x 1: of its window's first
    // element, counted from P rows and columns before the images; `outside` gets a bit for every tap that is in the padding.
    // (n_lo, v0: the tile's first image and its first column in that one)
    __device__ static __forceinline__ unsigned offset_of(int c, int v0, int n_lo, unsigned& outside)
    {
        if constexpr (LAYOUT == kRows) return (unsigned)(c * K * 4);
        const int v = v0 + c, img = v / OHWP, p = v % OHWP, y = (p / OW) * S, x = (p % OW) * S;
        const bool in = p < OHW && n_lo + img < NIMG;
        outside = in ? 0x80000000u : ~0u;
        if constexpr (P > 0)
#pragma unroll
            for (int t = 0; t < T; ++t)
                if (y + t / KW < P || y + t / KW >= H + P || x + t % KW < P || x + t % KW >= W + P) outside |= 1u << t;
        return in ? (unsigned)((img * CI * HW + y * W + x) * 4) : 0x7fffffffu;
    }
    __device__ static __forceinline__ auto rows_of(const float* A, int m0) { return __builtin_amdgcn_make_buffer_rsrc((void*)(A + (size_t)m0 * K), 0, BM * K * 4, 0x00020000); }
    __device__ static __forceinline__ auto columns_of(const float* B, long long n0, int n_lo)
    {
        return __builtin_amdgcn_make_buffer_rsrc(
            (void*)(LAYOUT == kRows ? B + (size_t)n0 * K : B + (size_t)n_lo * CI * HW - (P * W + P)), 0,
            LAYOUT == kRows ? BN * K * 4 : ((NIMG - n_lo < NIMAGES ? NIMG - n_lo : NIMAGES) * CI * HW + P * W + P) * 4, 0x00020000);
    }

    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        static_assert(FITS, "tile too large");
        const float* A = static_cast<const float*>(PREP ? Parts::source(I) : I);
        const float* B = static_cast<const float*>(F);
        float* __restrict__ C = static_cast<float*>(O);
        const int lane = tid & 63, li = lane & 15, kq = lane >> 4;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int g = wave / (WR * WN), w = wave % (WR * WN), wr = w / WN, wn = w % WN, gt = tid - g * GT;

        int mt, nt;
        if constexpr (LAYOUT == kRows) {
            // whole products are dealt to the XCDs, so that the tiles of one share an L2
            int batch = vblock / TILES, v = vblock % TILES;
            if constexpr (NIMG % 8 == 0) {
                const int xcd = vblock & 7, slot = vblock >> 3;
                batch = (slot / TILES) * 8 + xcd;
                v = slot % TILES;
            }
            mt = v / NT;
            nt = v % NT;
            A += (size_t)batch * M * K;
            B += (size_t)batch * W * K;
            C += (size_t)batch * M * W;
        } else {
            tile_of(vblock, nt, mt);
        }
        const int m0 = M % BM != 0 && mt == MT - 1 ? M - BM : mt * BM;
        const long long n0 = LAYOUT == kRows && W % BN != 0 && nt == NT - 1 ? W - BN : (long long)nt * BN;
        const int n_lo = LAYOUT == kRows ? 0 : (int)(n0 / OHWP);                 // kPix: first image of the tile
        const int v0 = (int)(n0 - (long long)n_lo * OHWP);

        auto column = [&](int c, unsigned& outside) { return offset_of(c, v0, n_lo, outside); };
        const auto ar = rows_of(A, m0);
        const auto br = columns_of(B, n0, n_lo);
        const unsigned a_voff = (unsigned)(((wr * TM * 16 + li) * K + 8 * kq) * 4);
        unsigned b_voff[NUB], b_out[NUB];
        int b_lds[NUB], b_k[NUB];
#pragma unroll
        for (int j = 0; j < NUB; ++j) {
            // threads past the last unit, or the last column of an octet, do another one again: the same values to the same place.  kRows: four lanes
            // read 128 consecutive bytes of a row; kPix: 64 lanes 64 consecutive columns of a plane
            const int u = (j * GT + gt) % (4 * BU), o = LAYOUT == kRows ? u & 3 : u / BU, cu = LAYOUT == kRows ? u >> 2 : u % BU;
            const int c = BU > BN && cu >= BN ? cu - 64 : cu;
            const unsigned v = column(c, b_out[j]);
            b_voff[j] = T > 1 || v == 0x7fffffffu ? v : v + 8 * o * B_K;
            b_k[j] = T > 1 ? __builtin_amdgcn_readfirstlane(8 * o) : 0;
            b_lds[j] = (o * BN + (TURNED ? c ^ 4 * o : c)) * 16;
        }

        f32x4 acc[TM][TN], part[TM][TN];            // the sum, and apart from it that of the last stages
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int b = 0; b < TN; ++b) acc[tm][b] = part[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};

        f32x4 ra[PREP ? 1 : TM][2];
        float rb[NUJ][8];
        unsigned pa[LEAN ? 1 : 2][TM][3][4];
        const auto pr = __builtin_amdgcn_make_buffer_rsrc((void*)(PREP ? Parts::block(I, m0 / 16) : nullptr), 0, PREP ? TM * WR * Parts::BLOCK_BYTES : 0, 0x00020000);
        // Taken apart before: the parts of stage s, straight into the registers that it is multiplied from.
        auto load_parts = [&](int set, int s) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(pr, (unsigned)(lane * 16 + q * 1024), ((wr * TM + tm) * NS + s) * 3072, 0));
#pragma unroll
                    for (int j = 0; j < 4; ++j) pa[LEAN ? 0 : set][tm][q][j] = v[j];
                }
        };
        auto load_a = [&](int tm, int s) {
            const unsigned v = TAIL != 0 && s == NS - 1 && 8 * kq >= TAIL ? 0x7fffffffu : a_voff;
#pragma unroll
            for (int h = 0; h < 2; ++h) ra[tm][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, v + (T > 1 ? 0 : h * 16), s * 128 + tm * 16 * K * 4 + (T > 1 ? h * 16 : 0), 0));
        };
        auto lds_of = [&](int j) { return EVEN ? b_lds[0] + j * (LAYOUT == kRows ? GT / 4 : GT / BU * BN) * 16 : b_lds[j]; };
        auto load_b = [&](int j, int s) {
            const int i = EVEN ? 0 : j;
            const unsigned v = T == 1 && TAIL != 0 && s == NS - 1 && lds_of(j) >= TAIL / 8 * BN * 16 ? 0x7fffffffu : b_voff[i];
            if constexpr (LAYOUT == kRows) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const f32x4 f = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(br, v + h * 16, s * 128 + (EVEN ? j * (GT / 4) * K * 4 : 0), 0));
#pragma unroll
                    for (int e = 0; e < 4; ++e) rb[j][4 * h + e] = f[e];
                }
            } else if constexpr (T > 1) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const unsigned at = TAPS.at[s * 32 + b_k[i] + (EVEN ? 8 * j * (GT / BU) : 0) + e];
                    // all ones (past the buffer) if this tap's bit is set; without padding only the last stage has such
                    const unsigned o = P > 0 || TAIL != 0 ? (unsigned)__builtin_amdgcn_sbfe((int)b_out[i], at, 1) : 0u;
                    rb[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, v | o, (at >> 5) * 4, 0));
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) rb[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, v, (s * 32 + (EVEN ? 8 * j * (GT / BU) : 0) + e) * B_K, 0));
            }
        };
        shared_with_asm(sm.t);
        unsigned char* const base = sm.t + g * NBUF * BUF;
        const unsigned char* const fb = base + (kq * BN + wn * TN * 16 + (TURNED ? li ^ 4 * kq : li)) * 16;
        unsigned pb[3][4];
        unsigned left = PREP ? Parts::inexact(I, m0 / 16 + wr * TM, TM, lane) : 0;   // see split.h
        if (tid == 0) sm.inexact = 0;
        // Two of a unit's eight values: units 0 .. NUJ - 1 are this thread's of B, the others its rows of A.
        auto convert = [&](int part, int to, int off) {
            const int u = part / 4, j = part % 4;
            if (j == 0) gather_left(left);
            if (u < NUJ) {
                split2(rb[u][2 * j], rb[u][2 * j + 1], pb[0][j], pb[1][j], pb[2][j], left);
                if (j == 3) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(base + off + q * PLANE + lds_of(u)) = u32x4{pb[q][0], pb[q][1], pb[q][2], pb[q][3]};
                }
            } else {
                const int tm = u - NUJ;
                unsigned(&p)[3][4] = pa[to][tm];
                split2(ra[tm][j / 2][2 * (j % 2)], ra[tm][j / 2][2 * (j % 2) + 1], p[0][j], p[1][j], p[2][j], left);
            }
        };
        constexpr int NPART = 4 * (LEAN || PREP ? NUJ : NUJ + TM);
        // A partial sum goes to the result between its last stage's MFMAs and the first ones of the next: every other block of columns,
        // over the two stages (2 TN blocks) that this leaves, so that the additions too are dealt between MFMAs (1024 x 4096 x 4096 158 us;
        // all in one stage 164).  Convolutions, whose padding takes registers, add a block right behind its last MFMAs (448 -> 384 channels
        // is 17 registers short otherwise beside a partner in a thread-fused workgroup; alone 0-1 %), and keep one address of A's rows.
        constexpr auto fold_at = [](int b) { return TN == 1 ? 0 : b == 0 ? 1 : T > 1 ? b + 1 : 2 * b; };
        constexpr auto folded = [fold_at](int at) { int n = 0; for (int b = 0; b < TN; ++b) n += at == SUMMED - 1 ? fold_at(b) < TN : at == 0 && fold_at(b) >= TN; return n; };
        auto fold = [&](int b) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) acc[tm][b] += part[tm][b];
        };
        const auto stage_of = [&](int it) { return (it < NIT ? it : NIT - 1) * KG + g; };   // past the end: the last one again

#pragma unroll
        for (int i = 0; i < 2 && i < NIT; ++i) {
#pragma unroll
            for (int j = 0; j < NUJ; ++j) load_b(j, stage_of(i));
            if constexpr (PREP) {
                if (i == 0) load_parts(0, g);
            } else if (i == 0) {
#pragma unroll
                for (int tm = 0; tm < TM; ++tm) load_a(tm, g);
            }
#pragma unroll
            for (int part = 0; part < 4 * NUJ; ++part) convert(part, 0, i * BUF);
        }
        if constexpr (NIT > 2)
#pragma unroll
            for (int j = 0; j < NUJ; ++j) load_b(j, stage_of(2));
        // A of the stage whose loads were the last; then those of stage `next`, if there is one
        auto convert_a = [&](int next, bool more) {
#pragma unroll
            for (int part = 4 * NUJ; part < 4 * (NUJ + TM); ++part) convert(part, 0, 0);
            if (more)
#pragma unroll
                for (int tm = 0; tm < TM; ++tm) load_a(tm, stage_of(next));
        };
        if constexpr (!LEAN && !PREP) convert_a(1, NIT > 1);
        u32x4 fr[2][3];
        auto read = [&](int set, int q, int b, int off) { fr[set][q] = *reinterpret_cast<const u32x4*>(fb + off + q * PLANE + b * 256); };
        sync.raw();
#pragma unroll
        for (int q = 2; q >= 0; --q) read(0, q, 0, 0);
        int off = 0, next = NIT > 1 ? BUF : 0, ahead = 2 * BUF;   // LDS offsets of this stage and the two after it
        // `at`: which one of the SUMMED stages of a partial sum this is.
        // `left`: how many stages follow, if those are less than three: nothing is loaded, taken apart or read past the last one.
        auto stage = [&](int it, auto at, auto left) {
            constexpr int AT = decltype(at)::value, FROM = AT % 2, LEFT = decltype(left)::value;
            constexpr int FIRST = LEFT >= 2 ? 0 : 4 * NUJ, LAST = LEAN || PREP || LEFT >= 1 ? NPART : 4 * NUJ, N = LAST > FIRST ? LAST - FIRST : 0;
            constexpr int VPM = (11 * N + (NIT > SUMMED ? 4 * TM * folded(AT) : 0) + 6 * TM * TN - 1) / (6 * TM * TN);
            // Behind the barrier the next stage is in LDS whole, and nobody reads the one before this any more.
            if (it > 0) sync.raw();
            if constexpr (LEAN) convert_a(it + 1, LEFT >= 1);
            if constexpr (PREP && LEFT >= 1) load_parts(FROM ^ 1, stage_of(it + 1));
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                const int set = (b + FROM * (TN & 1)) & 1;
#pragma unroll
                for (int t = 0; t < SplitTerms::N; ++t) {
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) {
                        const unsigned(&p)[4] = pa[LEAN ? 0 : FROM][tm][SplitTerms::A[t]];
                        const f32x4 c = AT == 0 && t == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : part[tm][b];
                        part[tm][b] = mfma_bf16(fr[set][SplitTerms::B[t]], u32x4{p[0], p[1], p[2], p[3]}, c);
                    }
                    if ((b + 1 < TN || LEFT >= 1) && t % 2 == 0) read(set ^ 1, 2 - t / 2, b + 1 < TN ? b + 1 : 0, b + 1 < TN ? off : next);
                }
#pragma unroll
                for (int i = FIRST; i < FIRST + N; ++i)
                    if ((i - FIRST) * TN / N == b) {
                        convert(i, LEAN ? 0 : FROM ^ 1, ahead);
                        if (i % 4 == 3) {
                            if (i / 4 < NUJ && LEFT >= 3) load_b(i / 4, stage_of(it + 3));
                            if (i / 4 >= NUJ && LEFT >= 2) load_a(i / 4 - NUJ, stage_of(it + 2));
                        }
                    }
                if (NIT > SUMMED && (AT == 0 || AT == SUMMED - 1)) {
                    const int when = AT == 0 ? TN + b : b;
#pragma unroll
                    for (int c = 0; c < TN; ++c)
                        if (when == fold_at(c)) fold(c);
                }
#pragma unroll
                for (int t = 0; t < SplitTerms::N; ++t) {
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // an MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);   // vector instructions
                    }
                    if ((b + 1 < TN || LEFT >= 1) && t % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            const int o = off;
            off = next;
            next = ahead;
            ahead = o;
            asm("" : "+s"(off), "+s"(next), "+s"(ahead));   // addresses are worked out anew: kept ones cost registers
        };
        // N stages, the last of all if END
        auto stages = [&](int it, auto n, auto end) {
            constexpr int N = decltype(n)::value, END = decltype(end)::value ? 0 : 3;
            if constexpr (N > 0) stage(it, std::integral_constant<int, 0>{}, std::integral_constant<int, END + N - 1>{});
            if constexpr (N > 1) stage(it + 1, std::integral_constant<int, 1>{}, std::integral_constant<int, END + N - 2>{});
            if constexpr (N > 2) stage(it + 2, std::integral_constant<int, 2>{}, std::integral_constant<int, END + N - 3>{});
            if constexpr (N > 3) stage(it + 3, std::integral_constant<int, 3>{}, std::integral_constant<int, END + N - 4>{});
        };
        // the last ones apart; of large tiles only those that the loop leaves, the compiler runs out of registers otherwise
        constexpr int REST = TM * TN <= 8 || NIT <= SUMMED ? (NIT - 1) % SUMMED + 1 : NIT % SUMMED;
#pragma unroll 1
        for (int it = 0; it + SUMMED <= NIT - REST; it += SUMMED) stages(it, std::integral_constant<int, SUMMED>{}, std::false_type{});
        stages(NIT - REST, std::integral_constant<int, REST>{}, std::true_type{});
#pragma unroll
        for (int b = 0; b < TN; ++b)
            if (NIT <= SUMMED || NIT % SUMMED != 0 || fold_at(b) >= TN) fold(b);

        // (the lane worked out again: three registers less in the loop)
        const int el = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), ei = el & 15, eq = el >> 4;
        if (split_inexact(left)) sm.inexact = 1;
        sync.raw();
        const bool again = sm.inexact != 0;
        if constexpr (KG > 1) {
            f32x4* const red = reinterpret_cast<f32x4*>(sm.t) + w * TM * TN * 64 + el;
            if (g > 0) {
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int b = 0; b < TN; ++b) red[((g - 1) * WR * WN * TM * TN + tm * TN + b) * 64] = acc[tm][b];
            }
            sync.raw();
            if (g > 0) return;
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int b = 0; b < TN; ++b)
#pragma unroll
                    for (int q = 1; q < KG; ++q) acc[tm][b] += red[((q - 1) * WR * WN * TM * TN + tm * TN + b) * 64];
        }
        finish(acc, again, A, B, C, m0, mt, n0, nt, n_lo, wr, wn, ei, eq, column, [&](int col, int& img, int& p) { return quad_at(v0 + col, n_lo, img, p); });
    }

    // kPix: the image and pixel of column v counted from image n_lo, and how many of it and the next three are one image's.
    __device__ static __forceinline__ int quad_at(int v, int n_lo, int& img, int& p)
    {
        img = n_lo + v / OHWP;
        p = v % OHWP;
        return img >= NIMG ? 0 : OHW - p < 4 ? OHW - p : 4;
    }

    // Lane (i, q) of 16 gets lane (i ^ 8, q)'s.
    __device__ static __forceinline__ float swap_halves(float v) { return dpp_mov<0x128>(v); }      // row_ror:8

    // What follows the sums of a wave: the results that three parts do not give are done again, and all are stored.
    // offset(c, outside): as offset_of, for column c of the tile; quad(c, img, p): as quad_at; QUADS: four columns are one image's and aligned; WHOLE: as LINES.
    template <bool QUADS = OHW % 4 == 0, bool WHOLE = LINES, class Offset, class Quad>
    __device__ static __forceinline__ void finish(f32x4 (&acc)[TM][TN], bool again, const float* A, const float* B, float* __restrict__ C, int m0, int mt, long long n0, int nt, int n_lo,
                                                  int wr, int wn, int ei, int eq, Offset offset, Quad quad)
    {
        const auto ar = rows_of(A, m0);
        const auto br = columns_of(B, n0, n_lo);
        // Which 16-row blocks are done again: all of the tile's, or the wave's with a result that is not finite (by block, so that the
        // bits do not depend on how many blocks a wave has).
        bool redo[TM], any = false;
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            float zero = 0.f;                       // or NaN
#pragma unroll
            for (int b = 0; b < TN; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) zero = __builtin_fmaf(acc[tm][b][v], 0.f, zero);
            redo[tm] = again || __builtin_amdgcn_ballot_w64(zero != 0.f) != 0;
            any |= redo[tm];
        }
        if (any) {
            // In ascending order of k, four an MFMA, as a sum that overflows wants it.
            f32x4 re[TM][TN];
            unsigned bo[TN], outside[TN];
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                const unsigned c = offset((wn * TN + b) * 16 + ei, outside[b]);
                bo[b] = LAYOUT == kRows ? c + eq * 16 : T > 1 || c == 0x7fffffffu ? c : c + eq * B_K;
            }
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int b = 0; b < TN; ++b) re[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (LAYOUT == kRows) {
                // Rows on both sides: group q of 16 lanes loads k + 4q .. k + 4q + 3 and gets k + q, k + 4 + q, .. from the others.
#pragma unroll 1
                for (int k = 0; k < K; k += 16) {
                    const bool past = K % 16 != 0 && k + 4 * eq >= K;
                    f32x4 a[TM], v[TN];
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
                        a[tm] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, past ? 0x7fffffffu : (unsigned)((((wr * TM + tm) * 16 + ei) * K + 4 * eq) * 4), k * 4, 0));
#pragma unroll
                    for (int b = 0; b < TN; ++b) v[b] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(br, past ? 0x7fffffffu : bo[b], k * 4, 0));
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) transpose_groups(a[tm]);
#pragma unroll
                    for (int b = 0; b < TN; ++b) transpose_groups(v[b]);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int b = 0; b < TN; ++b)
#pragma unroll
                            for (int tm = 0; tm < TM; ++tm) re[tm][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[b][e], a[tm][e], re[tm][b], 0, 0, 0);
                }
            } else {
                // Eight k at a time; the next eight are on their way meanwhile.
                float na[2][TM], nb[2][TN];
                auto fetch = [&](int k) {
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int tm = 0; tm < TM; ++tm)
                            na[e][tm] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ar, (((wr * TM + tm) * 16 + ei) * K + eq + 4 * e) * 4, k * 4, 0));
                    unsigned at[2];
                    if constexpr (T > 1) {
                        unsigned t[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) t[e] = TAPS.at[k + e];
#pragma unroll
                        for (int e = 0; e < 2; ++e) at[e] = eq & 2 ? (eq & 1 ? t[4 * e + 3] : t[4 * e + 2]) : (eq & 1 ? t[4 * e + 1] : t[4 * e]);
                    }
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int b = 0; b < TN; ++b) {
                            unsigned o = bo[b];
                            if constexpr (T > 1) {
                                o |= (unsigned)__builtin_amdgcn_sbfe((int)outside[b], at[e], 1);
                                if (o != ~0u) o += (at[e] >> 5) * 4;
                            }
                            nb[e][b] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, o, T > 1 ? 0 : (k + 4 * e) * B_K, 0));
                        }
                };
                fetch(0);
#pragma unroll 1
                for (int k = 0; k < K; k += 8) {
                    float a[2][TM], v[2][TN];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
#pragma unroll
                        for (int tm = 0; tm < TM; ++tm) a[e][tm] = na[e][tm];
#pragma unroll
                        for (int b = 0; b < TN; ++b) v[e][b] = nb[e][b];
                    }
                    fetch(k + 8 < K ? k + 8 : k);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int b = 0; b < TN; ++b)
#pragma unroll
                            for (int tm = 0; tm < TM; ++tm) re[tm][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e][b], a[e][tm], re[tm][b], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
                if (redo[tm])
#pragma unroll
                    for (int b = 0; b < TN; ++b) acc[tm][b] = re[tm][b];
        }
        if constexpr (WHOLE) {
            // Two blocks of columns and of eight rows at a time: lanes of rows 8 .. 15 have the second block's columns of the first rows and the other way round, so that
            // eight lanes write a line.
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int b = 0; b < TN; b += 2) {
                    f32x4 o[2];
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float x = ei < 8 ? acc[tm][b + 1][v] : acc[tm][b][v], y = swap_halves(x);
                        o[0][v] = ei < 8 ? acc[tm][b][v] : y;
                        o[1][v] = ei < 8 ? y : acc[tm][b + 1][v];
                    }
                    const int row = m0 + (wr * TM + tm) * 16 + (ei & 7), col = (wn * TN + b + (ei >> 3)) * 16 + 4 * eq;
                    int img = 0, p = 0;
                    if (LAYOUT == kRows || quad(col, img, p) > 0) {
                        float* const d = LAYOUT == kRows ? C + (size_t)row * W + n0 + col : C + ((size_t)img * M + row) * OHW + p;
#pragma unroll
                        for (int h = 0; h < 2; ++h) __builtin_nontemporal_store(o[h], reinterpret_cast<f32x4*>(d + (size_t)(8 * h) * (LAYOUT == kRows ? W : OHW)));
                    }
                }
            return;
        }
        // lane (i, q): row i of a 16-row block, columns 4q .. 4q + 3 of each 16-column block
        const auto own_row = [&](int m) { return M % BM == 0 || m >= mt * BM; };
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            const int col = (wn * TN + b) * 16 + 4 * eq;
            if constexpr (LAYOUT == kRows) {
#pragma unroll
                for (int tm = 0; tm < TM; ++tm) {
                    const int m = m0 + (wr * TM + tm) * 16 + ei;
                    if (own_row(m) && (W % BN == 0 || n0 + col >= nt * BN)) *reinterpret_cast<f32x4*>(C + (size_t)m * W + n0 + col) = acc[tm][b];
                }
            } else {
                int img, p;
                const int n = quad(col, img, p);
                if (n > 0) {
                    float* __restrict__ y = C + ((size_t)img * M + m0 + wr * TM * 16 + ei) * OHW + p;
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) {
                        if (!own_row(m0 + (wr * TM + tm) * 16 + ei)) continue;
                        float* const d = y + (size_t)(tm * 16) * OHW;
                        const f32x4 o = acc[tm][b];
                        if constexpr (QUADS) {
                            *reinterpret_cast<f32x4*>(d) = o;
                        } else if (n == 4) {
                            *reinterpret_cast<f32x4u*>(d) = f32x4u{o[0], o[1], o[2], o[3]};
                        } else {
#pragma unroll
                            for (int e = 0; e < 3; ++e)
                                if (e < n) d[e] = o[e];
                        }
                    }
                }
            }
        }
    }
};

// (see Narrow) us, ten waves and five, with twice the rows of a wave: 768 -> 160 channels on 17 x 17 460 and 514, 192 -> 320 at
// stride 2 385 and 436, 1280 -> 320 on 8 x 8 296 and 324, 2048 -> 320 459 and 500.  (Eight waves of 80 x 32: the 3 x 3 layer spills.)
template <int M, int K, int H, int W, int S, int NIMG, int TM, int WR, int WN, int KG, int BN, int LAYOUT, int KH, int KW, int P, bool LEAN, bool PREP, int LINES>
struct NarrowOf<GemmSplit<M, K, H, W, S, NIMG, TM, WR, WN, KG, BN, LAYOUT, KH, KW, P, LEAN, PREP, LINES>> {
    static constexpr int HALVE = 64 * WR * WN * KG > 512 && WR % 2 == 0 ? 2 : 1;
    using type = GemmSplit<M, K, H, W, S, NIMG, TM * HALVE, WR / HALVE, WN, KG, BN, LAYOUT, KH, KW, P, LEAN, PREP, LINES>;
};

}  // namespace bfuse
