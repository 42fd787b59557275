// Convolution of a batch as one implicit GEMM over large tiles: the throughput form of ConvF32Lds
// (ops_conv_general.h), for layers of at least 16 input channels with enough pixels in the batch to fill the chip.
//
// What bounded the per-wave form there: every wave staged a patch of its own through registers (address arithmetic,
// predicated scattered LDS writes) for 16 - 64 output channels, so the same image patch was staged CO / BM times, and
// tiles of 64 pixels per image leave a quarter of the lanes idle on 14 x 14 and 17 x 17 images.  37 - 110 TFLOP/s of
// the 154 the matrix cores sustain.  (Most layers of a batch have since gone on to the bf16 matrix cores, GemmSplit; ConvTiling says which
// stay: few workgroups, 64 output channels at stride 2, channel counts that its tiles do not divide.)  Here
//   * one workgroup of four waves owns BM output channels x BP consecutive pixels OF THE BATCH (a tile runs on into
//     the next image: no ragged tiles but the batch's last), each wave a (BM / WM) x (BP / WN) part of it;
//   * both operands of four input channels (a stage) are shared by the four waves: the filter rows, which are
//     contiguous in memory ([4 channels][T taps] per output channel), and the image patch, one plane per channel;
//   * both go from memory straight into LDS: the filter by 16-byte loads with a scalar base, the patch by 4-byte loads
//     whose per-lane offset (which image element belongs at this position of the patch) does not change from stage to
//     stage -- only a scalar offset moves on.  Padding and rows outside the image are lanes whose offset lies past the
//     buffer's end: they read as zero.  There is no vector instruction in the loop but LDS reads and MFMAs;
//   * two LDS buffers and one barrier per stage: the next stage lands while this one is multiplied (9 taps x 4
//     channels of a 128 x 128 tile are 144 MFMAs = 4600 clocks per wave).
//
// A operand (rows = output channels) of tap t: lane (i, q) reads A[i][q * T + t]: a row is
// 4 T words, for T = 9 the 64 lanes hit 64 banks.  B operand (columns = pixels): lane (i, q) reads plane
// q at the position of its pixel's window plus a compile-time offset per tap; the four planes start
// PLANE_BANK(q) banks apart so that lanes of different channels do not meet (stride 1: 16 consecutive words each;
// stride 2: 16 even words of 32; more: a word in four).
#pragma once
#include <hip/hip_runtime.h>

#include "dispatch.h"
#include "ops_conv_general.h"
#include "wave.h"

namespace bfuse {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// 64 lanes x 4 bytes straight to LDS from a raw buffer: lane L fetches base + soff + voff (zero if voff lies past the
// buffer), the data lands at lds_addr + 4 L.  `rsrc`, `soff` and `lds_addr` are wave-uniform.  Not counted by the
// compiler in vmcnt (see dma_load_lds_b128).
__device__ __forceinline__ void dma_buffer_lds_b32(unsigned voff, i32x4 rsrc, unsigned soff, unsigned lds_addr)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds"
                 :
                 : "v"(voff), "s"(rsrc), "s"(soff), "s"(lds_addr)
                 : "memory", "m0");
#endif
}

template <int CI_, int CO_, int H_, int W_, int KH_, int KW_, int S_, int P_, int BM_, int BP_, int WM_, int NIMG_>
struct ConvF32Tile {
    static constexpr bool MATRIX_CORES = true;   // the inner loop is a stream of MFMAs (what the fusion chooser asks)
    static constexpr int CI = CI_, CO = CO_, H = H_, W = W_, KH = KH_, KW = KW_, S = S_, P = P_, BM = BM_, BP = BP_, WM = WM_, NIMG = NIMG_;
    static constexpr int OH = (H - KH + 2 * P) / S + 1, OW = (W - KW + 2 * P) / S + 1;
    static constexpr int HW = H * W, OHW = OH * OW, T = KH * KW;
    static constexpr int NWAVE = 4, WN = NWAVE / WM;
    static constexpr int TM = BM / WM / 16, TN = BP / WN / 16;      // 16 x 16 blocks of a wave
    static constexpr int CPS = 4;                                   // channels of a stage: the four k of an MFMA, a plane per wave
    static constexpr int NS = CI / CPS;                             // stages
    // One accumulator over the whole reduction rounds after every four products of it: 256 -> 256 channels on 14 x 14 are
    // 5.8e-7 off (2-norm, against 64 bits) where the per-wave forms' four partial sums are 2.9e-7 off.  So the sum of every
    // SUM stages is added to a second set of registers (64 - 100 additions), three quarters as long as the parts those forms
    // give their waves (SUM_PARTS is the most of them): 2.6e-7.  The additions are nothing; the registers cost a workgroup
    // of the two to four on a CU, 1.64 -> 1.71 ms on that layer, 0-5 % on the others.
    static constexpr int SUM_PARTS = CI / 16 % 4 == 0 ? 4 : CI / 16 % 2 == 0 ? 2 : 1;
    static constexpr int SUM = 3 * NS / (4 * SUM_PARTS) > 1 ? 3 * NS / (4 * SUM_PARTS) : 1;
    static constexpr long long NPIX = (long long)OHW * NIMG;
    static constexpr long long TILES = (NPIX + BP - 1) / BP * (CO / BM);
    static constexpr int NPT = (int)((NPIX + BP - 1) / BP), NCT = CO / BM;
    static_assert(CI % CPS == 0 && CPS == NWAVE && CO % BM == 0 && BM % (16 * WM) == 0 && BP % (16 * WN) == 0, "channel tiling");
    static_assert((CI * T) % 4 == 0, "filter rows are whole 16-byte chunks");

    // ---- the patch: the image rows under the tile's output rows, image after image, every column a window touches.
    // Image n's rows are HR virtual rows (its OH windows' rows -P .. ), one image after the other.
    static constexpr int HR = (OH - 1) * S + KH, WPS = (OW - 1) * S + KW;
    static constexpr int MOST_LOADS = 28;                             // wave-level loads of a plane: a register each
    // The virtual rows that the BP pixels of the tile starting at pixel a span: S for every output row, and where one image
    // ends and the next begins KH - S more (windows of two images share no row; the least number of ends if that is negative).
    static constexpr long long rows_from(long long a)
    {
        return S * ((a % OW + BP - 1) / OW) + (KH - S) * (KH < S ? (BP - 1) / OHW : (a % OHW + BP - 1) / OHW) + KH;
    }
    // The most that any tile spans.  Rows depend on a tile's start within its output row, which comes round after at most OW
    // tiles, and ends on the tiles that hold one, which are alike after at most BP images (tiles of more than an image: all
    // of at most OHW different starts hold one).  Looking at these is exact and cheap; at all tiles of a large image it is
    // beyond what a compiler evaluates (512 x 512 pixels).
    static constexpr int patch_rows()
    {
        if (KH * WPS > 64 * MOST_LOADS) return KH;            // too wide to be staged at all: no need to look
        long long most = 0;
        const long long starts = BP > OHW ? OHW : OW;
        for (long long t = 0; t < starts && t * BP < NPIX; ++t)
            if (rows_from(t * BP) > most) most = rows_from(t * BP);
        for (long long n = 1; n < NIMG && n <= BP; ++n) {
            const long long a = (n * OHW - 1) / BP * BP;      // the tile that holds image n - 1's last pixel
            if (rows_from(a) > most) most = rows_from(a);
        }
        return (int)most;
    }
    static constexpr int NR = patch_rows();
    static constexpr int NIMAGES = (BP + OHW - 2) / OHW + 1;          // images a tile can touch
    static constexpr int NPOS = NR * WPS;
    static constexpr int NLB = (NPOS + 63) / 64;                     // wave-level loads per plane
    static constexpr int PLANE = NLB * 64;                            // words
    __host__ __device__ static constexpr int plane_bank(int q) { return S == 1 ? 16 * q : S == 2 ? 32 * (q / 2) + q % 2 : q; }
    static constexpr int A_CHUNKS = BM * CPS * T / 4;                // 16-byte chunks of the filter rows
    static constexpr int NLA = (A_CHUNKS + 63) / 64;
    static constexpr int A_BYTES = NLA * 1024;
    static constexpr int B_BYTES = (CPS * PLANE + 64) * 4;           // 64: the last plane starts up to 48 words late
    static constexpr int BUF = (A_BYTES + B_BYTES + 255) / 256 * 256;
    static constexpr int NLA_W = (NLA + NWAVE - 1) / NWAVE;          // per wave
    // fragment offsets are 16-bit immediates; two workgroups share a CU; the images of a tile are one buffer, whose size is 31
    // bits: an offset of 2^31 - 1 has to lie past its end
    static constexpr bool FITS = A_BYTES + B_BYTES < 65536 && 4 * BUF <= 160 * 1024 && NLB <= MOST_LOADS && TILES < (1LL << 31) &&
                                 (long long)(NIMAGES < NIMG ? NIMAGES : NIMG) * CI * HW * 4 < (1LL << 31);

    static constexpr Dims3 GRID{NPT * NCT, 1, 1};
    static constexpr Dims3 BLOCK{64 * NWAVE, 1, 1};
    static constexpr int THREADS = 64 * NWAVE;
    static constexpr bool HAS_BARRIERS = true;
    static constexpr bool LOOP_BARRIERS = true;
    static constexpr int MIN_BARRIERS = NS;

    struct Smem {
        __attribute__((aligned(1024))) unsigned char t[2 * BUF];
    };
    typedef __attribute__((address_space(3))) unsigned char lds_u8;

    // Workgroup id -> (pixel tile, output-channel tile): id % 8 is taken as the XCD, which owns consecutive pixel
    // tiles and every channel tile of each, so that the workgroups sharing a patch use one L2.
    __device__ static __forceinline__ void tile_of(int vblock, int& pt, int& ct)
    {
        constexpr int PER_XCD = NPT / 8;
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

    struct Ctx {
        unsigned a_voff[NLA_W], b_voff[NLB];
        const char* a_ub;        // filter rows of the tile, stage 0 (scalar)
        i32x4 rsrc;              // the images the tile touches
        unsigned lds;            // LDS byte address of buffer 0
        int wave;
    };
    __device__ static __forceinline__ void issue(const Ctx& c, int s, int buf)
    {
        const unsigned dst = c.lds + (unsigned)buf * BUF;
#pragma unroll
        for (int j = 0; j < NLA_W; ++j) {
            const int l = j * NWAVE + c.wave;
            if (NLA % NWAVE == 0 || l < NLA) dma_load_lds_b128(c.a_voff[j], c.a_ub + (size_t)s * (CPS * T * 4), dst + l * 1024);
        }
        const unsigned soff = (unsigned)(s * CPS + c.wave) * (unsigned)(HW * 4);
        const unsigned plane = dst + A_BYTES + (unsigned)(c.wave * PLANE + plane_bank(c.wave)) * 4u;
#pragma unroll
        for (int l = 0; l < NLB; ++l) dma_buffer_lds_b32(c.b_voff[l], c.rsrc, soff, plane + l * 256);
    }

    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        static_assert(FITS, "tile too large");
        const float* __restrict__ X = static_cast<const float*>(I);
        const float* __restrict__ Wt = static_cast<const float*>(F);
        float* __restrict__ Y = static_cast<float*>(O);
        int pt, ct;
        tile_of(vblock, pt, ct);
        const int co0 = ct * BM;
        const long long g0 = (long long)pt * BP;             // first pixel of the tile, over the batch
        const int n_lo = (int)(g0 / OHW), p_lo = (int)(g0 - (long long)n_lo * OHW);
        const int oy_lo = p_lo / OW;
        const int lane = tid & 63, li = lane & 15, kq = lane >> 4;

        Ctx c;
        c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        c.lds = (unsigned)(unsigned long long)(lds_u8*)sm.t;
        c.a_ub = reinterpret_cast<const char*>(Wt + (size_t)co0 * CI * T);
        {
            const unsigned long long base = (unsigned long long)(X + (size_t)n_lo * CI * HW);
            const int images = NIMG - n_lo < NIMAGES ? NIMG - n_lo : NIMAGES;
            c.rsrc = i32x4{(int)(unsigned)base, (int)(unsigned)(base >> 32), images * CI * HW * 4, 0x00020000};   // raw buffer, 32-bit elements
        }
#pragma unroll
        for (int j = 0; j < NLA_W; ++j) {
            int ch = (j * NWAVE + c.wave) * 64 + lane;
            if (ch >= A_CHUNKS) ch = A_CHUNKS - 1;           // lands in the slot's padding
            c.a_voff[j] = (unsigned)((ch / (CPS * T / 4)) * (CI * T) + (ch % (CPS * T / 4)) * 4) * 4u;
        }
        // which image element belongs at position lane + 64 l of a plane
#pragma unroll
        for (int l = 0; l < NLB; ++l) {
            const int pos = l * 64 + lane;
            const int v = pos / WPS + oy_lo * S, img = v / HR;
            const int iy = v % HR - P, ix = pos % WPS - P;
            const bool in = iy >= 0 && iy < H && ix >= 0 && ix < W && pos < NPOS && img < NIMAGES;
            c.b_voff[l] = in ? (unsigned)(img * CI * HW + iy * W + ix) * 4u : 0x7fffffffu;   // past the buffer: reads as zero
        }

        const int wm = c.wave / WN, wn = c.wave % WN;
        const unsigned char* ap = sm.t + ((wm * TM * 16 + li) * (CPS * T) + kq * T) * 4;
        const unsigned char* bp[TN];
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
            int q = p_lo + (wn * TN + tn) * 16 + li;                // pixel, counted from image n_lo's first
            if (g0 - p_lo + q > NPIX - 1) q = (int)(NPIX - 1 - (g0 - p_lo));   // past the batch: a valid address, the result is not stored
            const int img = q / OHW, p = q % OHW;
            const int pos = (img * HR + (p / OW - oy_lo) * S) * WPS + (p % OW) * S;
            bp[tn] = sm.t + A_BYTES + (kq * PLANE + plane_bank(kq) + pos) * 4;
        }

        f32x4 acc[TM][TN];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 sum[SUM < NS ? TM : 1][SUM < NS ? TN : 1] = {};
        int sum_at = SUM;

        issue(c, 0, 0);
        int step = BUF;
#pragma unroll 1
        for (int s = 0; s < NS; ++s) {
            // this wave's part of the stage has landed; behind the barrier everybody's has, and nobody reads the
            // other buffer any more
            __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
            sync.raw();
            if (s + 1 < NS) issue(c, s + 1, (s + 1) & 1);

            float a[2][TM], b[2][TN];
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) a[0][tm] = *reinterpret_cast<const float*>(ap + tm * 16 * CPS * T * 4);
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) b[0][tn] = *reinterpret_cast<const float*>(bp[tn]);
#pragma unroll
            for (int tap = 0; tap < T; ++tap) {
                if (tap + 1 < T) {
                    const int next = tap + 1;
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
                        a[next & 1][tm] = *reinterpret_cast<const float*>(ap + (tm * 16 * CPS * T + next) * 4);
#pragma unroll
                    for (int tn = 0; tn < TN; ++tn)
                        b[next & 1][tn] = *reinterpret_cast<const float*>(bp[tn] + ((next / KW) * WPS + next % KW) * 4);
                }
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int tn = 0; tn < TN; ++tn)
                        acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[tap & 1][tm], b[tap & 1][tn], acc[tm][tn], 0, 0, 0);
                // the next tap's reads one by one between this one's MFMAs
                if (tap + 1 < T) {
#pragma unroll
                    for (int r = 0; r < TM + TN; ++r) {
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                              // an LDS read
                        __builtin_amdgcn_sched_group_barrier(0x008, (TM * TN) / (TM + TN), 0);           // MFMAs
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            ap += step;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) bp[tn] += step;
            step = -step;
            if constexpr (SUM < NS) {
                if (s + 1 == sum_at) {
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                        for (int tn = 0; tn < TN; ++tn) {
                            sum[tm][tn] += acc[tm][tn];
                            acc[tm][tn] = f32x4{0.f, 0.f, 0.f, 0.f};
                        }
                    sum_at += SUM;
                }
            }
        }
        if constexpr (SUM < NS) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) acc[tm][tn] += sum[tm][tn];
        }

        // lane (j = pixel, rg) holds output channels 4 rg + v of a block
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) {
            const long long g = g0 + (wn * TN + tn) * 16 + li;
            if (g < NPIX) {
                const int img = (int)(g / OHW), p = (int)(g % OHW);
                float* __restrict__ y = Y + ((size_t)img * CO + co0 + wm * TM * 16 + 4 * kq) * OHW + p;
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int v = 0; v < 4; ++v) y[(size_t)(tm * 16 + v) * OHW] = acc[tm][tn][v];
            }
        }
    }
};

// The shared-tile form under ConvF32Lds's name: WM_ waves over the output channels, KS_ is the stage's channels, PB_ counts
// the workgroup's 16-pixel blocks as there.
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int BM, int PB, int NIMG>
struct ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, 4, NIMG, 1> : ConvF32Tile<CI, CO, H, W, KH, KW, S, P, BM, 16 * PB, 1, NIMG> {};
template <int CI, int CO, int H, int W, int KH, int KW, int S, int P, int BM, int PB, int NIMG>
struct ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, 4, NIMG, 2> : ConvF32Tile<CI, CO, H, W, KH, KW, S, P, BM, 16 * PB, 2, NIMG> {};

}  // namespace bfuse
