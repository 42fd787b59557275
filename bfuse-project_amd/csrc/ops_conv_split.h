// Convolution of a batch on the bf16 matrix cores whose images are taken apart once (see split.h): the form of GemmSplit for 3 x 3
// filters at stride 1.
//
//   Y[n][m][y][x] = sum over taps (i, j) and channels c of F[m][c][i][j] X[n][c][y S + i - P][x S + j - P]
//
// As a product whose second operand is gathered from the images (GemmSplit), every element is loaded, taken apart and written to LDS
// once for each tap it is under; on 256 -> 256 channels of 14 x 14, batch 1024, leaving out those loads and conversions and the filters' takes 1028 us to 671,
// and LDS writes alone are 300 of a stage's 3700 clocks (13 a wave and 16 bytes a lane).  Here
//   * the patch of 32 channels under a workgroup's tile (rows of the images one below the other, with their padding) is in LDS as
//     parts, [part][octet of channels][place][16 bytes]: a place is taken apart once, and the nine taps read it at nine offsets that are
//     immediates, since a step of a tap is the same number of places everywhere.  1.2 - 1.8 units of eight values for a column where the product takes
//     nine apart.  A row's wrap inside 16 columns costs a second LDS pass (2 % of the time);
//   * k counts (32 channels, tap), which is not how filters lie in memory, so they are put in that order by a kernel that runs before
//     this one (SplitParts: 5 - 10 us) and takes them apart on that occasion: a lane's 48 bytes of a tap and 16 rows are three coalesced loads
//     straight into the registers that are multiplied from, a tap ahead;
//   * two LDS buffers and one barrier for 32 channels, that is for nine times 12 TN MFMAs of a wave; the units of the next channels are loaded and
//     taken apart between them, one at a time;
//   * tiles of four waves (32 rows each) of which two fit a CU's LDS, so that one multiplies where the other waits: 128 x 112 columns on 28 x 28
//     images take 945 us, 256 columns on eight waves 1019.  Where consecutive pixels make the patch too large (wide images have whole rows above and below), the tile is a
//     rectangle of one image; ConvTiling has the choice.
//
// Batch 1024, us, GemmSplit and now, both in turn on one card, uniform operands: 256 -> 256 on 14 x 14 1109 -> 901, 128 on 28 x 28 1179 -> 945, 512 on 7 x 7
// 1227 -> 977, 448 -> 384 on 8 x 8 953 -> 758, 96 on 35 x 35 1228 -> 990, 64 -> 96 909 -> 701, 64 on 56 x 56 1599 -> 1199, 64 -> 128 without padding 2306 ->
// 1993, 128 -> 256 on 28 x 28 likewise 1785 -> 1728, 32 -> 64 on 147 x 147 6210 -> 4500: 1.24x in the
// geometric mean.  256 -> 256 is 263 of the 335 TFLOP/s that six bf16 MFMAs for a product leave on random operands.  Of its 900 us the filters' parts
// cost 64, the patch 47 and wraps 20; the MFMAs and their LDS reads alone take 758 (650 on constant operands).
// The counters have the matrix cores busy 0.82 of the time at 1.73 GHz (GemmSplit: 0.61 at 1.86), so power bounds it; 64 on 56 x 56, with 1.4 vector instructions an
// MFMA instead of 0.5, 0.54 at 1.98.
//
// Sums: a partial sum of one, two or three taps (of 32 channels each) is added to the result's: the longer it is the more error it has, the shorter
// the more of them are added, which large results feel most.  Errors against 64 bits on images after a ReLU, three sets of operands, GemmSplit's and
// these, 2-norm and largest over the results' rms: 256 -> 256 1.73e-7 -> 1.56e-7 and 1.49e-6 -> 1.60e-6, 512 1.89 -> 1.76 and 1.92 -> 2.00, 448 -> 384 1.85 -> 1.70 and 1.77 ->
// 1.85, 128 1.61 -> 1.24 and 1.47 -> 1.37, 96 1.55 -> 1.16 and 1.44 -> 1.25, 64 -> 96 1.09 -> 1.08 and 1.13 -> 1.17, 64 on 56 x 56 1.09 -> 1.08 and 1.16 -> 1.20, 64 -> 128 1.10 ->
// 1.09 and 1.16 -> 1.26, 128 -> 256 1.59 -> 1.24 and 1.46 -> 1.41, 32 -> 64 0.98 -> 0.72 and 1.34 -> 1.05.  So the 2-norm is smaller at all ten layers, the largest
// up to 1.08 times at six of them.  Other lengths: 32 channels by two taps 0.98 and 1.38 (2.5 % faster), 64 by one 0.92 and 1.33, 128 by three 1.41 and 1.36,
// 256 by two 1.51 and 1.90.  What three parts do not hold is done again as there.
#pragma once
#include <hip/hip_runtime.h>

#include <numeric>
#include <type_traits>
#include <utility>

#include "dispatch.h"
#include "ops_gemm_split.h"
#include "split.h"
#include "wave.h"

namespace bfuse {

// I: the filters' parts (SplitParts), F: the images.  TM, WR, WN, BN: as in GemmSplit.
template <int CI_, int CO_, int H_, int W_, int KH_, int KW_, int S_, int P_, int NIMG_, int TM_, int WR_, int WN_, int BN_, int TW_ = 0>
struct ConvSplit {
    using Form = GemmSplit<CO_, CI_ * KH_ * KW_, H_, W_, S_, NIMG_, TM_, WR_, WN_, 1, BN_, kPix, KH_, KW_, P_>;
    using Parts = SplitParts<CO_, CI_ * KH_ * KW_, KH_ * KW_>;
    static constexpr int PARTS_OPERAND = 0;
    static constexpr bool MATRIX_CORES = true;
    static constexpr int CI = CI_, CO = CO_, H = H_, W = W_, KH = KH_, KW = KW_, S = S_, P = P_, NIMG = NIMG_, TM = TM_, WR = WR_, WN = WN_, BN = BN_;
    static constexpr int T = KH * KW, NG = CI / 32, THREADS = Form::THREADS, BM = Form::BM, TN = Form::TN, OW = Form::OW, OHW = Form::OHW, OHWP = Form::OHWP;
    // TW > 0: the tile is a rectangle of an image, TW pixels wide.  Otherwise its pixels follow each other in the batch, and the patch has the
    // images, with their padding, one below the other: the rows of the tile's output rows, and KH - S more for every image that follows the first.
    static constexpr int TW = TW_, TH = TW > 0 ? BN / TW : 1, TX = TW > 0 ? (OW + TW - 1) / TW : 1, TY = TW > 0 ? (Form::OH + TH - 1) / TH : 1;
    static_assert(TW == 0 || (BN % TW == 0 && TW % 4 == 0), "rectangle");
    static constexpr int NT = TW > 0 ? TX * TY * NIMG : Form::NT;
    static constexpr int PH = (Form::OH - 1) * S + KH, PW = ((TW > 0 ? TW : OW) - 1) * S + KW;
    // Of images of up to 8192 pixels the most that a tile has from any place where one begins.
    static constexpr int STEP = std::gcd(BN, OHWP);
    static constexpr int NIMAGES = TW > 0 ? 1 : (BN + OHWP - STEP - 1) / OHWP + 1;
    static constexpr int rows_from(int v) { return (v + BN - 1) / OHWP * PH + ((v + BN - 1) % OHWP < OHW ? (v + BN - 1) % OHWP : OHW - 1) / OW * S - v / OW * S + KH; }
    static constexpr int pick_rows()
    {
        if (TW > 0) return (TH - 1) * S + KH;
        if (OHWP > 8192) return (NIMAGES - 1) * (KH > S ? KH - S : 0) + (BN + OW - 2) / OW * S + KH;
        int most = 0;
        for (int v = 0; v < OHWP; v += STEP) most = rows_from(v) > most ? rows_from(v) : most;
        return most;
    }
    static constexpr int ROWS = pick_rows();
    // A rectangle's blocks of 16 columns come round after whole rows: ROW_STEP places further down.
    static constexpr int PERIOD = TW > 0 ? TW / std::gcd(TW, 16) : TN, NAT = PERIOD < TN ? PERIOD : TN, ROW_STEP = TW > 0 ? NAT * 16 / (TW > 0 ? TW : 1) * S * PW : 0;
    static constexpr int SLOTS = ROWS * PW, UNITS = 4 * SLOTS;                       // places, units (eight channels of a place) of 32 channels
    static constexpr int NUJ = (UNITS + THREADS - 1) / THREADS;
    // The taps at which unit j of the next channels is loaded and taken apart, at least one later: a thread has the values of one unit at a
    // time, so that where units are many the next one's loads follow the conversions of the same tap.
    static constexpr int load_at(int j) { return 2 * NUJ <= T ? j * T / NUJ : j * T / (NUJ + 1); }
    static constexpr int apart_at(int j) { return 2 * NUJ <= T ? (j + 1) * T / NUJ - 1 : (j + 1) * T / (NUJ + 1); }
    static constexpr int unit_of(bool load, int t) { for (int j = 0; j < NUJ; ++j) if ((load ? load_at(j) : apart_at(j)) == t) return j; return -1; }
    static constexpr int PLANE = UNITS * 16, BUF = 3 * PLANE, NBUF = NG > 1 ? 2 : 1;
    static_assert(TN > 1, "a partial sum is added to the result beside the next block of columns");
    static constexpr int SUMMED = NG == 1 ? 1 : NG * T <= 36 ? 2 : 3;                // taps of a partial sum (see Sums)
    static constexpr bool FITS = Form::FITS && CI % 32 == 0 && T > 1 && NBUF * BUF <= 163840 - 256 && (NG > 1 ? NUJ < T : NUJ <= 12) && (long long)BM * CI * T * 6 < (1LL << 31);
    static constexpr long long TILES = (long long)NT * Form::MT;
    static constexpr Dims3 GRID{(int)TILES, 1, 1}, BLOCK = Form::BLOCK;
    static constexpr bool HAS_BARRIERS = true, LOOP_BARRIERS = true;
    static constexpr int MIN_BARRIERS = NG;

    struct Smem {
        __attribute__((aligned(16))) unsigned char t[NBUF * BUF];
        unsigned inexact;
    };

    template <class Fn, int... t>
    __device__ static __forceinline__ void each(Fn fn, std::integer_sequence<int, t...>)
    {
        (fn(std::integral_constant<int, t>{}), ...);
    }
    // Has the value here: additions that are needed only behind the loop go there otherwise, and what they add stays in registers.
    __device__ static __forceinline__ void pin(f32x4& v)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" : "+v"(v));
#endif
    }

    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        static_assert(FITS, "tile");
        const float* A = static_cast<const float*>(Parts::source(I));
        const float* B = static_cast<const float*>(F);
        const int lane = tid & 63, li = lane & 15, kq = lane >> 4;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave / WN, wn = wave % WN;
        int mt, nt;
        Form::template tile_of<NT>(vblock, nt, mt);
        const int m0 = CO % BM != 0 && mt == Form::MT - 1 ? CO - BM : mt * BM;
        // the tile's first image, in it the first column (rectangles: output row and column), and the patch's first row and column there
        const long long n0 = (long long)nt * BN;
        const int n_lo = TW > 0 ? nt / (TX * TY) : (int)(n0 / OHWP), v0 = TW > 0 ? 0 : (int)(n0 - (long long)n_lo * OHWP);
        const int ty = TW > 0 ? nt / TX % TY * TH : 0, tx = TW > 0 ? nt % TX * TW : 0;
        const int r0 = TW > 0 ? ty * S : v0 / OW * S, x0 = tx * S;

        // The units of a thread: u is the channels 8 (u / SLOTS) .. of place u % SLOTS.  Those past the last one are done twice, with the
        // same values to the same place.
        const auto br = __builtin_amdgcn_make_buffer_rsrc((void*)(B + (size_t)n_lo * CI * H * W), 0, (NIMG - n_lo < NIMAGES ? NIMG - n_lo : NIMAGES) * CI * H * W * 4, 0x00020000);
        unsigned b_voff[NUJ];
        auto unit = [&](int j) { const int u = j * THREADS + tid; return j == NUJ - 1 && UNITS % THREADS != 0 && u >= UNITS ? u % UNITS : u; };
#pragma unroll
        for (int j = 0; j < NUJ; ++j) {
            const int u = unit(j), place = u % SLOTS, row = r0 + place / PW, img = TW > 0 ? 0 : row / PH, y = row - img * PH - P, x = x0 + place % PW - P;
            const bool in = y >= 0 && y < H && x >= 0 && x < W && n_lo + img < NIMG && img < NIMAGES;
            b_voff[j] = in ? (unsigned)(((img * CI + u / SLOTS * 8) * H * W + y * W + x) * 4) : 0x7fffffffu;
        }
        const int b_lds = unit(0) * 16, b_last = unit(NUJ - 1) * 16;
        // where this lane's columns find their window's first place
        unsigned at[NAT];
        shared_with_asm(sm.t);
#pragma unroll
        for (int b = 0; b < NAT; ++b) {
            const int c = (wn * TN + b) * 16 + li, v = v0 + c, img = v / OHWP, p = v % OHWP < OHW ? v % OHWP : OHW - 1;
            const int place = TW > 0 ? c / (TW > 0 ? TW : 1) * S * PW + c % (TW > 0 ? TW : 1) * S : n_lo + img < NIMG ? (img * PH + p / OW * S - r0) * PW + p % OW * S : 0;
            at[b] = (unsigned)((kq * SLOTS + place) * 16);
        }

        const auto pr = __builtin_amdgcn_make_buffer_rsrc((void*)Parts::block(I, m0 / 16), 0, BM / 16 * Parts::BLOCK_BYTES, 0x00020000);
        unsigned pa[2][TM][3][4];
        unsigned left = Parts::inexact(I, m0 / 16 + wr * TM, TM, lane);
        int s_off = wr * TM * Parts::BLOCK_BYTES, c_off = 0;        // bytes to the parts and the channels that are loaded next
        auto load_parts = [&](int set, int s) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(pr, (unsigned)(lane * 16 + q * 1024), s + tm * Parts::BLOCK_BYTES, 0));
#pragma unroll
                    for (int j = 0; j < 4; ++j) pa[set][tm][q][j] = v[j];
                }
        };
        float rb[NUJ][8];
        auto load_unit = [&](int j, int r, int c) {
#pragma unroll
            for (int e = 0; e < 8; ++e) rb[r][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, b_voff[j], c + e * (H * W * 4), 0));
        };
        unsigned pb[3][4];
        auto convert = [&](int j, int r, int part, int off) {
            if (part == 0) gather_left(left);
            split2(rb[r][2 * part], rb[r][2 * part + 1], pb[0][part], pb[1][part], pb[2][part], left);
            if (part == 3) {
                unsigned char* const to = sm.t + off + (j == NUJ - 1 && UNITS % THREADS != 0 ? b_last : b_lds + j * THREADS * 16);
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(to + q * PLANE) = u32x4{pb[q][0], pb[q][1], pb[q][2], pb[q][3]};
            }
        };
        if (tid == 0) sm.inexact = 0;
#pragma unroll
        for (int j = 0; j < NUJ; ++j) load_unit(j, j, 0);
        load_parts(0, s_off);
#pragma unroll
        for (int j = 0; j < NUJ; ++j)
#pragma unroll
            for (int part = 0; part < 4; ++part) convert(j, j, part, 0);

        f32x4 acc[TM][TN], part[TM][TN];            // the sum, and apart from it that of the last taps
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int b = 0; b < TN; ++b) acc[tm][b] = part[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto fold = [&](int b) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) {
                acc[tm][b] += part[tm][b];
                pin(acc[tm][b]);
            }
        };
        u32x4 fr[2][3];
        int off = 0;
        auto read = [&](int set, int q, int b, int t) { fr[set][q] = *reinterpret_cast<const u32x4*>(sm.t + at[b % NAT] + q * PLANE + (b / NAT * ROW_STEP + t / KW * PW + t % KW) * 16); };
        sync.raw();
        // Tap t of 32 channels; `more`: others follow, whose images are taken apart meanwhile.
        auto tap = [&](auto t_, auto more_) {
            constexpr int t = decltype(t_)::value, AT = t % SUMMED, SET = t & 1;
            constexpr bool MORE = decltype(more_)::value, LAST = t == T - 1, ENDS = AT == SUMMED - 1 || LAST;
            constexpr int j0 = unit_of(true, t), j1 = unit_of(false, t);    // loaded now, taken apart now
            constexpr int CB = j0 >= 0 ? TN / 2 : TN;                        // the blocks of columns whose MFMAs it is taken apart beside
            constexpr int VPM = ((MORE && j1 >= 0 ? 50 : 0) + 4 * TM * TN / (ENDS ? 1 : TN) + 6 * TM * TN - 1) / (6 * TM * TN);
            if constexpr (!LAST || MORE) {
                s_off += 3072;
                load_parts(SET ^ 1, s_off);
            }
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                const int set = (b + t * TN) & 1;
#pragma unroll
                for (int i = 0; i < SplitTerms::N; ++i) {
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) {
                        const unsigned(&p)[4] = pa[SET][tm][SplitTerms::A[i]];
                        const f32x4 c = AT == 0 && i == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : part[tm][b];
                        part[tm][b] = mfma_bf16(fr[set][SplitTerms::B[i]], u32x4{p[0], p[1], p[2], p[3]}, c);
                    }
                    if ((b + 1 < TN || !LAST) && i % 2 == 0) read(set ^ 1, 2 - i / 2, b + 1 < TN ? b + 1 : 0, b + 1 < TN ? t : t + 1);
                }
                if constexpr (MORE && j1 >= 0) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (i * CB / 4 == b) convert(j1, 0, i, BUF - off);
                }
                if constexpr (MORE && j0 >= 0)
                    if (b == (j1 >= 0 ? CB : 0)) load_unit(j0, 0, c_off);
                // a partial sum goes to the result a block of columns behind its last MFMAs
                if (ENDS && b > 0) fold(b - 1);
                if (b == 0 && AT == 0 && t > 0) fold(TN - 1);
#pragma unroll
                for (int i = 0; i < SplitTerms::N; ++i) {
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // an MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);   // vector instructions
                    }
                    if ((b + 1 < TN || !LAST) && i % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (LAST) fold(TN - 1);
        };
        auto group = [&](auto more) {
            c_off += 32 * H * W * 4;
#pragma unroll
            for (int q = 2; q >= 0; --q) read(0, q, 0, 0);
            each([&](auto t) { tap(t, more); }, std::make_integer_sequence<int, T>{});
            if constexpr (decltype(more)::value) {
                if constexpr (T % 2 != 0)
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
#pragma unroll
                            for (int j = 0; j < 4; ++j) pa[0][tm][q][j] = pa[1][tm][q][j];
                const int step = BUF - 2 * off;
#pragma unroll
                for (int b = 0; b < NAT; ++b) {
                    at[b] += step;
#if defined(__HIP_DEVICE_COMPILE__)
                    asm("" : "+v"(at[b]));           // kept, and nothing made of it
#endif
                }
                off += step;
                // Behind the barrier the next channels are in LDS whole, and nobody reads these any more.
                sync.raw();
            }
        };
#pragma unroll 1
        for (int g = 0; g + 1 < NG; ++g) group(std::true_type{});
        group(std::false_type{});

        const int el = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
        if (split_inexact(left)) sm.inexact = 1;
        sync.raw();
        auto rectangle = [&](int c, int& y, int& x) {
            y = ty + c / (TW > 0 ? TW : 1);
            x = tx + c % (TW > 0 ? TW : 1);
            return y < Form::OH && x < OW;
        };
        if constexpr (TW > 0) {
            Form::template finish<OW % 4 == 0, false>(acc, sm.inexact != 0, A, B, static_cast<float*>(O), m0, mt, n0, nt, n_lo, wr, wn, el & 15, el >> 4,
                [&](int c, unsigned& outside) {
                    int y, x;
                    const bool in = rectangle(c, y, x);
                    return Form::offset_of(in ? y * OW + x : OHW, 0, n_lo, outside);
                },
                [&](int c, int& img, int& p) {
                    int y, x;
                    const bool in = rectangle(c, y, x);
                    img = n_lo;
                    p = y * OW + x;
                    return in ? (OW - x < 4 ? OW - x : 4) : 0;
                });
        } else {
            Form::finish(acc, sm.inexact != 0, A, B, static_cast<float*>(O), m0, mt, n0, nt, n_lo, wr, wn, el & 15, el >> 4,
                [&](int c, unsigned& outside) { return Form::offset_of(c, v0, n_lo, outside); }, [&](int c, int& img, int& p) { return Form::quad_at(v0 + c, n_lo, img, p); });
        }
    }
};

// (see Slim) Waves of 16 rows, twice as many, read every fragment for half the MFMAs.
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int NIMG, int TM, int WR, int WN, int BN, int TW>
struct SlimOf<ConvSplit<CI, CO, H, W, KH, KW, S, P, NIMG, TM, WR, WN, BN, TW>> {
    using type = ConvSplit<CI, CO, H, W, KH, KW, S, P, NIMG, 1, TM * WR, WN, BN, TW>;
};

}  // namespace bfuse
