// fp32 matrix product on large tiles that four waves share: the throughput form of GemmF32 (ops_gemm_f32.h: batched
// products) and of Conv1x1F32 (ops_conv_1x1.h), for problems with enough tiles to fill the chip.
//
//   C[m][n] = sum_k A[m][k] * B(k, n)
//
// The per-wave forms load every operand of a wave's tile for that wave alone, through its registers; they run one
// wave per SIMD (more only queue in the memory pipeline) and leave the matrix cores idle whenever it waits: 59 - 118
// TFLOP/s, or 2 - 3.2 TB/s where the bytes count, of 154 and 4.7.  Here a workgroup stages BM rows of A and BN columns
// of B for KS steps of k in LDS, memory -> LDS directly, in NBUF buffers (loads NBUF - 1 stages ahead) with one barrier
// per stage: nothing but LDS reads and MFMAs in the loop, and two or more workgroups share a CU.  126 - 142 TFLOP/s where
// the matrix cores bound it, 3.8 - 5.1 TB/s where memory does.  Since GemmSplit took the
// long reductions over (bf16 matrix cores, 160 - 240 TFLOP/s) it keeps products of few channels: 1 x 1 layers of fewer than 256, which
// memory bounds or whose tiles are mostly ends, and the 16-head scores at batch 1.  (A single dense product is better off on
// GemmF32Ring, 150 TFLOP/s against 131-143 here: with one or two tiles per CU no second workgroup hides a stage's barrier.)
//
// A rows are contiguous along k: [BM][KS] in LDS, 16-byte chunk c of row r at c ^ f(r) so that the 16 rows of a
// fragment read spread over the banks.  Lane (i, q) reads A[i][16g + 4q .. +3] with one 128-bit read: element t is
// the operand of MFMA step t of the 16-k group g, which sums over the lanes' k = 16g + 4q + t.
// B comes in one of two layouts:
//   kPix    planes of n for each k (an image batch [NIMG][K][HW], n = a pixel; a [K, N] matrix is one image of N
//           pixels): [KS][BN] in LDS.  Lane (j, q) reads 4 consecutive columns of plane 16g + 4q + t at once; element
//           e goes to accumulator block e of the 64-column group, whose column j is 4j + e: a lane ends up with four
//           consecutive columns and stores 16 bytes.  Columns are counted over the batch with every image rounded up
//           to whole chunks of 4 pixels, so that no chunk belongs to two images (289 pixels: 1 % more columns).
//           Pixels of a strided layer are fetched one by one (4-byte loads), others in 16-byte chunks.
//   kRows   rows of B contiguous along k, [N][K]: staged like A, lane (j, q) reads B[4j + e][16g + 4q .. +3].
// A row tile (kRows: also a column tile) that does not divide the problem starts BM rows (BN columns) before its end:
// it overlaps its neighbour and both write the same bits (see GemmF32).
#pragma once
#include <hip/hip_runtime.h>

#include "dispatch.h"
#include "ops_conv_tile.h"
#include "wave.h"

namespace bfuse {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));   // 16 bytes on a 4-byte boundary

enum BLayout : int { kPix = 0, kRows = 1 };

// 64 lanes x 16 bytes straight to LDS from a raw buffer (see dma_buffer_lds_b32)
__device__ __forceinline__ void dma_buffer_lds_b128(unsigned voff, i32x4 rsrc, unsigned soff, unsigned lds_addr)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :
                 : "v"(voff), "s"(rsrc), "s"(soff), "s"(lds_addr)
                 : "memory", "m0");
#endif
}

// M, K: rows of A and their length.  kPix: H x W images, stride S, NIMG of them (a [K, N] matrix: 1 x N, 1, 1);
// kRows: W is N, NIMG the number of independent products (H = S = 1).
template <int M_, int K_, int H_, int W_, int S_, int NIMG_, int BM_, int BN_, int WM_, int KS_, int LAYOUT_, int NBUF_ = 2>
struct GemmTile {
    static constexpr bool MATRIX_CORES = true;   // the inner loop is a stream of MFMAs (what the fusion chooser asks)
    static constexpr int M = M_, K = K_, H = H_, W = W_, S = S_, NIMG = NIMG_, BM = BM_, BN = BN_, WM = WM_, KS = KS_, LAYOUT = LAYOUT_, NBUF = NBUF_;
    static constexpr int NWAVE = 4, WN = NWAVE / WM, THREADS = 64 * NWAVE;
    static constexpr int TM = BM / WM / 16, TG = BN / WN / 64, TN = 4 * TG;     // 16-row blocks, 64-column groups, 16-column blocks of a wave
    static constexpr int NS = K / KS, NG = KS / 16;                              // stages, 16-k groups of a stage
    // Products along rows with a long reduction sum 256 k at a time into a second set of registers, the halves that the
    // per-wave form gives two waves: 512 x 512 x 64 is 2.9e-7 off (2-norm, against 64 bits), with one sum 4.1e-7.
    static constexpr int SUM = LAYOUT == kRows && K >= 512 ? 256 / KS : NS;
    static constexpr int OH = (H - 1) / S + 1, OW = (W - 1) / S + 1, HW = H * W, OHW = OH * OW;
    static constexpr int OHWP = (OHW + 3) / 4 * 4;                               // columns of an image
    static constexpr int MT = (M + BM - 1) / BM;
    static constexpr int NT = LAYOUT == kRows ? (W + BN - 1) / BN : (int)(((long long)OHWP * NIMG + BN - 1) / BN);
    static constexpr bool GATHER = LAYOUT == kPix && S > 1;
    static_assert(BM % (16 * WM) == 0 && BN % (64 * WN) == 0 && K % KS == 0 && (KS == 16 || KS == 32), "tile");
    static_assert(M >= BM && (LAYOUT == kPix || (W >= BN && H == 1 && S == 1)), "a tile is not larger than the problem");
    static constexpr int NIMAGES = LAYOUT == kRows ? 1 : (BN + OHWP - 2) / OHWP + 1;   // images a tile can touch
    // The rows of a product, and the images of a tile, are addressed by 31 bits: columns past the batch (and past a strided
    // image) are read through an offset of 2^31 - 1, which has to lie past the end of the buffer that the images are.
    static constexpr bool FITS = (long long)M * K * 4 < (1LL << 31) && (long long)(NIMAGES < NIMG ? NIMAGES : NIMG) * K * HW * 4 < (1LL << 31);

    static constexpr int TILES = MT * NT;
    static constexpr Dims3 GRID{LAYOUT == kRows ? TILES * NIMG : TILES, 1, 1};
    static constexpr Dims3 BLOCK{THREADS, 1, 1};
    static constexpr bool HAS_BARRIERS = true;
    static constexpr bool LOOP_BARRIERS = true;
    static constexpr int MIN_BARRIERS = NS;

    // loads per wave and stage: the same number for every wave (waits count them), so A's space is whole rounds of loads
    static constexpr int A_W = (BM * KS * 4 + NWAVE * 1024 - 1) / (NWAVE * 1024), A_BYTES = A_W * NWAVE * 1024;
    static constexpr int B_BYTES = BN * KS * 4, BUF = A_BYTES + B_BYTES;
    static constexpr int B_W = (GATHER ? B_BYTES / 256 : B_BYTES / 1024) / NWAVE;
    static constexpr int LPS = A_W + B_W;
    static_assert(BUF < 65536 && B_BYTES % (NWAVE * 1024) == 0 && (NBUF - 2) * LPS <= 63 && (NBUF == 2 || NBUF == 3), "fragment offsets are 16-bit immediates");
    static constexpr int RC = KS / 4;                                            // 16-byte chunks of a row

    struct Smem {
        __attribute__((aligned(1024))) unsigned char t[NBUF * BUF];
    };
    typedef __attribute__((address_space(3))) unsigned char lds_u8;

    // where chunk c of row r lies: fragment reads of A take 16 consecutive rows, those of a kRows B every fourth row
    __device__ static __forceinline__ int swz_a(int r) { return RC == 8 ? (r >> 1) & 7 : (r >> 2) & 3; }
    __device__ static __forceinline__ int swz_b(int r) { return RC == 8 ? (r >> 2) & 7 : (r >> 2) & 3; }

    // kPix: (column tile, row tile), dealt so that the row tiles of one column tile follow each other on one XCD
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

    struct Ctx {
        const char *a_ub, *b_ub;                    // stage 0 of the tile's rows (scalar)
        i32x4 rsrc;                                 // kPix: the images the tile touches
        unsigned a_voff[A_W];
        unsigned b_voff[LAYOUT == kRows ? B_W : GATHER ? BN / 64 : 1];
        unsigned lds;
        int wave;
    };
    __device__ static __forceinline__ void issue(const Ctx& c, int s, int off)
    {
        const unsigned dst = c.lds + (unsigned)off;
#pragma unroll
        for (int j = 0; j < A_W; ++j) dma_load_lds_b128(c.a_voff[j], c.a_ub + (size_t)s * (KS * 4), dst + (j * NWAVE + c.wave) * 1024);
#pragma unroll
        for (int j = 0; j < B_W; ++j) {
            const int l = j * NWAVE + c.wave;
            if constexpr (LAYOUT == kRows) {
                dma_load_lds_b128(c.b_voff[j], c.b_ub + (size_t)s * (KS * 4), dst + A_BYTES + l * 1024);
            } else if constexpr (GATHER) {
                constexpr int LPP = BN / 64;         // loads per plane; a wave takes whole planes
                const int plane = (j / LPP) * NWAVE + c.wave;
                dma_buffer_lds_b32(c.b_voff[j % LPP], c.rsrc, (unsigned)(s * KS + plane) * (unsigned)(HW * 4), dst + A_BYTES + (plane * LPP + j % LPP) * 256);
            } else {
                // BN = 256: a load is one plane; 128: two; 64: four
                dma_buffer_lds_b128(c.b_voff[0], c.rsrc, (unsigned)(s * KS + l * (256 / BN)) * (unsigned)(HW * 4), dst + A_BYTES + l * 1024);
            }
        }
    }

    template <int N_OUT>
    __device__ static __forceinline__ void wait_vm()
    {
        __builtin_amdgcn_s_waitcnt((N_OUT & 0xF) | ((N_OUT >> 4) << 14) | 0x0F70);
    }

    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        static_assert(FITS, "tile too large");
        static_assert(LAYOUT == kRows || 256 % BN == 0, "a load is whole planes");
        const float* __restrict__ A = static_cast<const float*>(I);
        const float* __restrict__ B = static_cast<const float*>(F);
        float* __restrict__ C = static_cast<float*>(O);
        const int lane = tid & 63, li = lane & 15, kq = lane >> 4;
        Ctx c;
        c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        c.lds = (unsigned)(unsigned long long)(lds_u8*)sm.t;
        const int wm = c.wave / WN, wn = c.wave % WN;

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

        c.a_ub = reinterpret_cast<const char*>(A + (size_t)m0 * K);
#pragma unroll
        for (int j = 0; j < A_W; ++j) {
            int u = (j * NWAVE + c.wave) * 64 + lane;
            if (u >= BM * RC) u = BM * RC - 1;                              // past the tile: lands in the slot's padding
            const int r = u / RC;
            c.a_voff[j] = (unsigned)(r * K + ((u % RC) ^ swz_a(r)) * 4) * 4u;
        }
        int n_lo = 0;                                                       // kPix: first image of the tile
        if constexpr (LAYOUT == kRows) {
            c.b_ub = reinterpret_cast<const char*>(B + (size_t)n0 * K);
#pragma unroll
            for (int j = 0; j < B_W; ++j) {
                const int u = (j * NWAVE + c.wave) * 64 + lane, r = u / RC;
                c.b_voff[j] = (unsigned)(r * K + ((u % RC) ^ swz_b(r)) * 4) * 4u;
            }
        } else {
            n_lo = (int)(n0 / OHWP);
            const int images = NIMG - n_lo < NIMAGES ? NIMG - n_lo : NIMAGES;
            const unsigned long long base = (unsigned long long)(B + (size_t)n_lo * K * HW);
            c.rsrc = i32x4{(int)(unsigned)base, (int)(unsigned)(base >> 32), images * K * HW * 4, 0x00020000};   // raw buffer, 32-bit elements
            const int v0 = (int)(n0 - (long long)n_lo * OHWP);
            if constexpr (GATHER) {
#pragma unroll
                for (int l = 0; l < BN / 64; ++l) {
                    const int v = v0 + l * 64 + lane, img = v / OHWP, p = v % OHWP;
                    c.b_voff[l] = p < OHW && n_lo + img < NIMG ? (unsigned)(img * K * HW + (p / OW) * S * W + (p % OW) * S) * 4u : 0x7fffffffu;
                }
            } else {
                const int plane = lane / (BN / 4), v = v0 + (lane % (BN / 4)) * 4, img = v / OHWP, p = v % OHWP;
                // a chunk past the batch reads as zero; one that runs past its image reads on into the next plane: not stored
                c.b_voff[0] = n_lo + img < NIMG ? (unsigned)(img * K * HW + plane * HW + p) * 4u : 0x7fffffffu;
            }
        }

        // fragment addresses in buffer 0; group g of a row is chunk 4g + q, wherever the row's swizzle puts it
        const unsigned char* ap[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) ap[g] = sm.t + (wm * TM * 16 + li) * (KS * 4) + (((4 * g + kq) ^ swz_a(li)) * 16);
        const unsigned char* bp[LAYOUT == kRows ? NG : 1];
        if constexpr (LAYOUT == kRows) {
#pragma unroll
            for (int g = 0; g < NG; ++g) bp[g] = sm.t + A_BYTES + (wn * TG * 64 + 4 * li) * (KS * 4) + (((4 * g + kq) ^ swz_b(4 * li)) * 16);
        } else {
            bp[0] = sm.t + A_BYTES + (4 * kq * BN + wn * TG * 64 + 4 * li) * 4;
        }

        f32x4 acc[TM][TN];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int b = 0; b < TN; ++b) acc[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 sum[SUM < NS ? TM : 1][SUM < NS ? TN : 1] = {};
        int sum_at = SUM;

#pragma unroll
        for (int s = 0; s < NBUF - 1; ++s)
            if (s < NS) issue(c, s, s * BUF);
        int off = 0, ahead = (NBUF - 1) * BUF;     // LDS offsets of stage s and of stage s + NBUF - 1
#pragma unroll 1
        for (int s = 0; s < NS; ++s) {
            // this wave's part of the stage has landed; behind the barrier everybody's has, and nobody reads the stage before
            if (NBUF == 2 || s + NBUF - 1 > NS) wait_vm<0>();
            else wait_vm<(NBUF - 2) * LPS>();
            sync.raw();
            if (s + NBUF - 1 < NS) issue(c, s + NBUF - 1, ahead);

            f32x4 a[2][TM], b[2][LAYOUT == kRows ? TN : TG];
            auto read_a = [&](int g, int tm) { return *reinterpret_cast<const f32x4*>(ap[g] + off + tm * 16 * KS * 4); };
            // kRows: block u of group g, four k; kPix: 64-column group u of plane 16 (st / 4) + 4 q + st % 4
            auto read_b = [&](int st, int u) {
                if constexpr (LAYOUT == kRows) return *reinterpret_cast<const f32x4*>(bp[st] + off + ((u / 4) * 64 + u % 4) * KS * 4);
                else return *reinterpret_cast<const f32x4*>(bp[0] + off + (((st / 4) * 16 + st % 4) * BN + u * 64) * 4);
            };
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) a[0][tm] = read_a(0, tm);
            if constexpr (LAYOUT == kRows) {
#pragma unroll
                for (int u = 0; u < TN; ++u) b[0][u] = read_b(0, u);
            } else {
#pragma unroll
                for (int u = 0; u < TG; ++u) b[0][u] = read_b(0, u);
            }
#pragma unroll
            for (int g = 0; g < NG; ++g) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    // the next step's plane, and a quarter of the next group's fragments
                    int reads = 0;
                    if constexpr (LAYOUT == kPix) {
                        if (4 * g + t + 1 < 4 * NG) {
#pragma unroll
                            for (int u = 0; u < TG; ++u) b[(t + 1) & 1][u] = read_b(4 * g + t + 1, u);
                            reads += TG;
                        }
                    }
                    if (g + 1 < NG) {
#pragma unroll
                        for (int tm = 0; tm < TM; ++tm)
                            if (tm % 4 == t) {
                                a[(g + 1) & 1][tm] = read_a(g + 1, tm);
                                ++reads;
                            }
                        if constexpr (LAYOUT == kRows) {
#pragma unroll
                            for (int u = 0; u < TN; ++u)
                                if (u % 4 == t) {
                                    b[(g + 1) & 1][u] = read_b(g + 1, u);
                                    ++reads;
                                }
                        }
                    }
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                        for (int u = 0; u < TN; ++u)
                            acc[tm][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[g & 1][tm][t], LAYOUT == kRows ? b[g & 1][u][t] : b[t & 1][u / 4][u % 4],
                                                                              acc[tm][u], 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 8; ++r)
                        if (r < reads) {
                            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
                            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);   // MFMAs
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            off = off == (NBUF - 1) * BUF ? 0 : off + BUF;
            ahead = ahead == (NBUF - 1) * BUF ? 0 : ahead + BUF;
            if constexpr (SUM < NS) {
                if (s + 1 == sum_at) {
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                        for (int b = 0; b < TN; ++b) {
                            sum[tm][b] += acc[tm][b];
                            acc[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};
                        }
                    sum_at += SUM;
                }
            }
        }
        if constexpr (SUM < NS) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int b = 0; b < TN; ++b) acc[tm][b] += sum[tm][b];
        }

        // lane (j, rg): rows 4 rg + v, columns 4j .. 4j + 3 of each 64-column group
#pragma unroll
        for (int g = 0; g < TG; ++g) {
            const int col = wn * TG * 64 + g * 64 + 4 * li;
            if constexpr (LAYOUT == kRows) {
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        f32x4 o;
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] = acc[tm][4 * g + e][v];
                        *reinterpret_cast<f32x4*>(C + (size_t)(m0 + wm * TM * 16 + tm * 16 + 4 * kq + v) * W + n0 + col) = o;
                    }
            } else {
                const int vc = (int)(n0 - (long long)n_lo * OHWP) + col, img = n_lo + vc / OHWP, p = vc % OHWP;
                if (img < NIMG) {
                    float* __restrict__ y = C + ((size_t)img * M + m0 + wm * TM * 16 + 4 * kq) * OHW + p;
                    const bool whole = OHW % 4 == 0 || p + 4 <= OHW;
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            f32x4 o;
#pragma unroll
                            for (int e = 0; e < 4; ++e) o[e] = acc[tm][4 * g + e][v];
                            float* const d = y + (size_t)(tm * 16 + v) * OHW;
                            if constexpr (OHW % 4 == 0) {
                                *reinterpret_cast<f32x4*>(d) = o;
                            } else if (whole) {
                                *reinterpret_cast<f32x4u*>(d) = f32x4u{o[0], o[1], o[2], o[3]};
                            } else {
#pragma unroll
                                for (int e = 0; e < 3; ++e)
                                    if (p + e < OHW) d[e] = o[e];
                            }
                        }
                }
            }
        }
    }
};

}  // namespace bfuse
