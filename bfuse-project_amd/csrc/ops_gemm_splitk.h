// fp32 GEMM side on the bf16 matrix cores (split.h), the waves of a workgroup splitting K: C[M,N] = A[M,K] . B[K,N] (+ optional
// tanh-GELU), for the problems of GemmF32Dma (ops_gemm_f32_dma.h), which have no more than one or two tiles of 4-5 thousand
// results for a CU -- too small for operands that waves share (GemmSplit).
//
// Every wave multiplies the whole tile over its own k-range, 32 k a stage, and takes both operands apart in its registers: no LDS
// and no barrier until the partial tiles meet.  Lane (i, q) loads A[i][8q .. 8q + 7] of a 16-row block, and B[8q + e][4i .. 4i + 3]
// (e = 0 .. 7) of a 64-column group, whose component c is its part of column block c, the columns 4i + c: a lane ends up with four
// consecutive columns of four rows.  A trailing group of 16 columns is loaded by single floats.  While a column block is
// multiplied the next one is taken apart; what a group was loaded into takes its next stage as soon as the last block has been.
//
// What bounds it is the wave's issue: an MFMA takes 10 clocks of it (it lasts 16) and a vector instruction 4.4, and a 32 x 144 tile
// has 108 of these and 528 of those a stage where the fp32 form has 144 MFMAs of 32.6: 3400 against 4700 clocks.  On tiles of fewer
// uses for every element it is no faster: us, fp32 ring before, 32 x 144 512 x 768 x 2304 15.9 -> 14.0-14.7 and 1024 x 768 x 2304 29.3 ->
// 24.5-25.8, 32 x 128 1024 x 4096 x 1024 61 -> 52-56, 32 x 96 two workgroups a CU 512 x 768 x 3072 20.4 -> 18.4-19.2; but 32 x 96 one
// workgroup a CU 1024 x 3072 x 768 39.2 -> 39.7, 32 x 64 512 x 4096 x 1024 37.0 -> 36.9, 32 x 48 512 x 3072 x 768 23.2 -> 23.6.  Fused:
// with the LayerNorm 16.1 -> 14.1-14.5, with the softmax (32 x 96, GELU) 22.6 -> 22.0, with LayerNorm and softmax 19.2 -> 16.6-17.2, with the 56 x 56 convolution 19.9 -> 17.2.  Eight waves
// of half the k (two a SIMD): 17.1 against 15.8; their partial tiles cost what their overlap gives.
//
// One sum over a wave's stages, rounded six times for every 32 k where the fp32 form rounds eight times: 2-norm errors against 64
// bits 2.0e-7 (K = 768) and 4.9e-7 (4096) where that one has 2.5e-7 and 5.8e-7.
//
// What three bf16 cannot hold (split.h): a wave whose sums are not all finite, or that has met a value that is more than its
// parts, hands over NaN.  Finite sums add up to NaN never, so all waves then see NaN in what they finish, and all multiply
// their k-range again with the fp32 instructions (512 x 768 x 2304: 16.6 us without such a value, 32-34 with; 39-41 with four
// dependent k at a time).
#pragma once
#include <hip/hip_runtime.h>

#include "dispatch.h"
#include "ops_gemm_f32.h"
#include "split.h"
#include "wave.h"

namespace bfuse {

// ROUNDS: row blocks' partial sums meet in LDS all at once, or in so many rounds of a part of it.
template <int M_, int N_, int K_, int BM_, int BN_, int KS_, int EPI_, int ROUNDS_>
struct GemmSplitK {
    static constexpr bool MATRIX_CORES = true;   // the inner loop is a stream of MFMAs (what the fusion chooser asks)
    static constexpr int M = M_, N = N_, K = K_, BM = BM_, BN = BN_, KS = KS_, EPI = EPI_, ROUNDS = ROUNDS_;
    static constexpr int TM = BM / 16, G4 = BN / 64, G1 = BN % 64 / 16, NB = 4 * G4 + G1;   // row blocks, 64- and 16-column groups, column blocks
    static constexpr int KW = K / KS, NS = KW / 32;                                          // k of a wave, its stages
    static_assert(G4 > 0 && M % BM == 0 && N % BN == 0 && KW % 32 == 0 && BM % 16 == 0 && BN % 16 == 0 && N % 4 == 0, "tile must divide the problem");
    static constexpr bool FITS = (long long)K * N * 4 < (1LL << 31) && (long long)BM * K * 4 < (1LL << 31);
    static constexpr Dims3 GRID{N / BN, M / BM, 1};
    static constexpr Dims3 BLOCK{64 * KS, 1, 1};
    static constexpr int THREADS = 64 * KS;
    static constexpr bool HAS_BARRIERS = KS > 1;
    static constexpr int TMR = TM / ROUNDS;                      // row blocks whose sums meet at a time
    static constexpr int UNIT = 64 * (16 * G4 + 4 * G1);         // bytes of component v of a row block's accumulators
    static constexpr int WAVE_BYTES = TMR * 4 * UNIT;
    static_assert(TM % ROUNDS == 0, "rounds");

    struct Smem {
        __attribute__((aligned(16))) unsigned char t[KS > 1 ? KS * WAVE_BYTES : 16];
    };

    __device__ static __forceinline__ float epilogue(float v)
    {
        if constexpr (EPI == kEpiGeluTanh) return gelu_tanh(v);
        return v;
    }

    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        static_assert(FITS, "operands are addressed by 31 bits");
        const float* A = static_cast<const float*>(I);
        const float* B = static_cast<const float*>(F);
        float* __restrict__ C = static_cast<float*>(O);
        const Dims3 vb = XcdTiles<N / BN, M / BM, BM, BN>::tile(vblock);
        const int m0 = vb.y * BM, n0 = vb.x * BN;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, kq = lane >> 4;
        const int kbeg = wave * KW;
        const auto ar = __builtin_amdgcn_make_buffer_rsrc((void*)(A + (size_t)m0 * K + kbeg), 0, (BM * K - kbeg) * 4, 0x00020000);
        const auto br = __builtin_amdgcn_make_buffer_rsrc((void*)(B + (size_t)kbeg * N + n0), 0, ((K - kbeg) * N - n0) * 4, 0x00020000);
        const unsigned a_voff = (unsigned)((li * K + 8 * kq) * 4), b_voff = (unsigned)((8 * kq * N + 4 * li) * 4), t_voff = (unsigned)((8 * kq * N + G4 * 64 + li) * 4);

        f32x4 acc[TM][NB];
        f32x4 ra[TM][2], rb[G4 > 0 ? G4 : 1][8];
        float rt[G1 > 0 ? G1 : 1][8];
        auto load_a = [&](int s) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int h = 0; h < 2; ++h) ra[tm][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ar, a_voff + (tm * 16 * K * 4 + h * 16), s * 128, 0));
        };
        // 64-column group g, or 16-column group g - G4
        auto load_b = [&](int g, int s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (g < G4) rb[g][e] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(br, b_voff + g * 256, (s * 32 + e) * (N * 4), 0));
                else rt[g - G4][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, t_voff + (g - G4) * 64, (s * 32 + e) * (N * 4), 0));
            }
        };
        unsigned pa[TM][3][4], pb[2][3][4];
        unsigned left = 0;                                  // see split.h
        auto convert_a = [&](int tm) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                split2(ra[tm][j / 2][2 * (j % 2)], ra[tm][j / 2][2 * (j % 2) + 1], pa[tm][0][j], pa[tm][1][j], pa[tm][2][j], left);
                gather_left(left);
            }
        };
        auto convert_b = [&](int b) {
            unsigned(&p)[3][4] = pb[b & 1];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float lo = b < 4 * G4 ? rb[b / 4 < G4 ? b / 4 : 0][2 * j][b % 4] : rt[b < 4 * G4 ? 0 : b - 4 * G4][2 * j];
                const float hi = b < 4 * G4 ? rb[b / 4 < G4 ? b / 4 : 0][2 * j + 1][b % 4] : rt[b < 4 * G4 ? 0 : b - 4 * G4][2 * j + 1];
                split2(lo, hi, p[0][j], p[1][j], p[2][j], left);
                gather_left(left);
            }
        };
        const auto group_of = [](int b) constexpr { return b < 4 * G4 ? b / 4 : G4 + b - 4 * G4; };

#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        load_a(0);
#pragma unroll
        for (int g = 0; g < G4 + G1; ++g) load_b(g, 0);
#pragma unroll 1
        for (int s = 0; s < NS; ++s) {
            const int ahead = s + 1 < NS ? s + 1 : s;       // past the end: the last one again
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) convert_a(tm);
            load_a(ahead);
            convert_b(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if (b + 1 < NB) convert_b(b + 1);
                // a group's registers are free once its last block has been taken apart
                if (b + 1 < NB && (b + 2 == NB || group_of(b + 2) != group_of(b + 1))) load_b(group_of(b + 1), ahead);
#pragma unroll
                for (int t = 0; t < SplitTerms::N; ++t)
#pragma unroll
                    for (int tm = 0; tm < TM; ++tm) {
                        const unsigned(&p)[4] = pa[tm][SplitTerms::A[t]];
                        const unsigned(&q)[4] = pb[b & 1][SplitTerms::B[t]];
                        acc[tm][b] = mfma_bf16(u32x4{p[0], p[1], p[2], p[3]}, u32x4{q[0], q[1], q[2], q[3]}, acc[tm][b]);
                    }
#pragma unroll
                for (int r = 0; r < 6 * TM; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                          // an MFMA
                    __builtin_amdgcn_sched_group_barrier(0x002, (46 + 6 * TM - 1) / (6 * TM), 0);   // vector instructions
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        float zero = 0.f;                                   // or NaN
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) zero = __builtin_fmaf(acc[tm][b][v], 0.f, zero);
        const float poison = __builtin_amdgcn_ballot_w64(split_inexact(left) || zero != 0.f) != 0 ? __builtin_nanf("") : 0.f;

        // component v of row block tm (row 4 rg + v of it) is unit 4 tm + v, finished by wave unit % KS
        unsigned char* const part = sm.t + lane * 16;
        unsigned char* const part1 = sm.t + G4 * 1024 + lane * 4;
        auto hand_over = [&](int r, float add) {
#pragma unroll
            for (int tm = 0; tm < TMR; ++tm)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int at = wave * WAVE_BYTES + (tm * 4 + v) * UNIT;
                    const f32x4(&a)[NB] = acc[r * TMR + tm];
#pragma unroll
                    for (int g = 0; g < G4; ++g) *reinterpret_cast<f32x4*>(part + at + g * 1024) = f32x4{a[4 * g][v], a[4 * g + 1][v], a[4 * g + 2][v], a[4 * g + 3][v]} + add;
#pragma unroll
                    for (int g = 0; g < G1; ++g) *reinterpret_cast<float*>(part1 + at + g * 256) = a[4 * G4 + g][v] + add;
                }
        };
        constexpr int NU = TMR * 4 / KS;                    // units a wave finishes
        static_assert(TMR * 4 % KS == 0, "every wave finishes as many rows");
        f32x4 o4[NU][G4 > 0 ? G4 : 1];
        float o1[NU][G1 > 0 ? G1 : 1];
        // the partial sums in wave order; whether one of them is NaN
        auto total = [&]() {
            float nan = 0.f;
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                const int u = i * KS + wave;
#pragma unroll
                for (int g = 0; g < G4; ++g) {
                    f32x4 o = *reinterpret_cast<const f32x4*>(part + u * UNIT + g * 1024);
#pragma unroll
                    for (int w = 1; w < KS; ++w) o += *reinterpret_cast<const f32x4*>(part + w * WAVE_BYTES + u * UNIT + g * 1024);
                    o4[i][g] = o;
                    nan = nan != nan ? nan : o[0];
                }
#pragma unroll
                for (int g = 0; g < G1; ++g) {
                    float o = *reinterpret_cast<const float*>(part1 + u * UNIT + g * 256);
#pragma unroll
                    for (int w = 1; w < KS; ++w) o += *reinterpret_cast<const float*>(part1 + w * WAVE_BYTES + u * UNIT + g * 256);
                    o1[i][g] = o;
                    nan = nan != nan ? nan : o;
                }
            }
            return __builtin_amdgcn_ballot_w64(nan != nan) != 0;
        };
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            if (r > 0) sync();                              // the sums before these have been read
            hand_over(r, r == 0 ? poison : 0.f);
            sync();
            if (total() && r == 0) {
                sync();
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};
                // Eight k at a time, in ascending order as a sum that overflows wants it; the next eight are on their way meanwhile.
                float na[2][TM];
                f32x4 nb[2][G4];
                float nt[2][G1 > 0 ? G1 : 1];
                auto fetch = [&](int k) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
#pragma unroll
                        for (int tm = 0; tm < TM; ++tm)
                            na[e][tm] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ar, (unsigned)(((tm * 16 + li) * K + kq + 4 * e) * 4), k * 4, 0));
#pragma unroll
                        for (int g = 0; g < G4; ++g)
                            nb[e][g] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(br, (unsigned)((kq * N + g * 64 + 4 * li) * 4), (k + 4 * e) * (N * 4), 0));
#pragma unroll
                        for (int g = 0; g < G1; ++g)
                            nt[e][g] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, (unsigned)((kq * N + G4 * 64 + g * 16 + li) * 4), (k + 4 * e) * (N * 4), 0));
                    }
                };
                fetch(0);
#pragma unroll 1
                for (int k = 0; k < KW; k += 8) {
                    float a[2][TM];
                    f32x4 v[2][G4];
                    float w[2][G1 > 0 ? G1 : 1];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
#pragma unroll
                        for (int tm = 0; tm < TM; ++tm) a[e][tm] = na[e][tm];
#pragma unroll
                        for (int g = 0; g < G4; ++g) v[e][g] = nb[e][g];
#pragma unroll
                        for (int g = 0; g < G1; ++g) w[e][g] = nt[e][g];
                    }
                    fetch(k + 8 < KW ? k + 8 : k);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int b = 0; b < NB; ++b)
#pragma unroll
                            for (int tm = 0; tm < TM; ++tm)
                                acc[tm][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e][tm], b < 4 * G4 ? v[e][b / 4 < G4 ? b / 4 : 0][b % 4] : w[e][b < 4 * G4 ? 0 : b - 4 * G4], acc[tm][b], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                hand_over(0, 0.f);
                sync();
                (void)total();
            }
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                const int u = i * KS + wave;
                float* __restrict__ row = C + (size_t)(m0 + (r * TMR + u / 4) * 16 + 4 * kq + u % 4) * N + n0;
#pragma unroll
                for (int g = 0; g < G4; ++g) {
                    f32x4 o = o4[i][g];
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = epilogue(o[e]);
                    *reinterpret_cast<f32x4*>(row + g * 64 + 4 * li) = o;
                }
#pragma unroll
                for (int g = 0; g < G1; ++g) row[G4 * 64 + g * 16 + li] = epilogue(o1[i][g]);
            }
        }
    }
};

}  // namespace bfuse
