// fp32 GEMM side on the bf16 matrix cores (split.h), the waves of a workgroup splitting K: C[M,N] = A[M,K] . B[K,N] (+ optional
// tanh-GELU), for the problems of GemmF32Dma (ops_gemm_f32_dma.h), which have no more than one or two tiles of 4-5 thousand
// results for a CU -- too small for operands that waves share (GemmSplit).
//
// Every wave multiplies the whole tile over its own k-range, 32 k a stage, and takes both operands apart in its registers; no barrier
// until the partial tiles meet.  B goes to registers: lane (i, q) loads B[8q + e][4i .. 4i + 3] (e = 0 .. 7) of a 64-column group, whose
// component c is its part of column block c, the columns 4i + c: a lane ends up with four consecutive columns of four rows.  The 16, 32
// or 48 columns past the last group are loaded one, two or three wide.  A goes to LDS, a place of the wave's own for one stage,
// by loads that need no register: its rows are what the lanes of an MFMA hold side by side, and a load in which neighbouring lanes
// want different rows takes the CU's address unit 64 clocks where eight lanes a row take 16 (measured; 32-row tiles: half of what the loop's
// loads took).  A stage's A is read into MFMA layout and taken apart at its top, the loads of the next go out behind that.
//
// While a column block is multiplied the next one is taken apart: part 0 beside the first half of the MFMAs, parts 1 and 2, into
// the registers that this leaves, beside the second.  What a group was loaded into takes its next stage as soon as its last block has been.
//
// What bounds it is the wave's issue: an MFMA takes 10 clocks of it (it lasts 16) and a vector instruction 4.4, and a 32 x 144 tile
// has 108 of these and 528 of those a stage where the fp32 form has 144 MFMAs of 32.6.  On tiles of fewer
// uses for every element it is no faster: us, fp32 ring before, 32 x 144 512 x 768 x 2304 15.9 -> 13.7-14.7 and 1024 x 768 x 2304 29.3 ->
// 24.5-25, 32 x 96 two workgroups a CU 512 x 768 x 3072 20.4 -> 17.0-17.5; but 32 x 48 512 x 3072 x 768 20.0 -> 20.6.  A in registers as well, loaded in
// MFMA layout, and all parts of a column block at once took 14.9-15.4 and 18.3-19.9, and 189 and 237 registers instead of 154 and 202: three workgroups a CU
// instead of two beside other operators.  Fused, before and now: 512 x 768 x 3072 with the softmax (GELU) 22.0 -> 20.0, with the 32-head products 35.5 and 37.4 -> 30.0 and 33.0,
// with the 56 x 56 convolution 21.3 -> 20.7; 512 x 768 x 2304 with the LayerNorm 14.2 -> 13.9, with scores of 12 heads 19.4 -> 18.2 (thread-fused
// with the 28 x 28 convolution 19.4 -> 19.9).  Eight waves of half the k on 32 x 144: 14.5 against 14.7; their partial tiles cost what their overlap gives.
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

#include <type_traits>

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
    static constexpr int TM = BM / 16, G4 = BN / 64, R = BN % 64 / 16, NB = 4 * G4 + R;     // row blocks, 64-column groups, 16-column blocks past them, column blocks
    static constexpr int KW = K / KS, NS = KW / 32;                                          // k of a wave, its stages
    static_assert(NB > 1 && M % BM == 0 && N % BN == 0 && KW % 32 == 0 && BM % 16 == 0 && BN % 16 == 0 && N % 4 == 0, "tile must divide the problem");
    static constexpr bool FITS = (long long)K * N * 4 < (1LL << 31) && (long long)BM * K * 4 < (1LL << 31);
    static constexpr Dims3 GRID{N / BN, M / BM, 1};
    static constexpr Dims3 BLOCK{64 * KS, 1, 1};
    static constexpr int THREADS = 64 * KS;
    static constexpr bool HAS_BARRIERS = KS > 1;
    static constexpr int TMR = TM / ROUNDS;                      // row blocks whose sums meet at a time
    static constexpr int UNIT = 64 * (16 * G4 + 4 * R);          // bytes of component v of a row block's accumulators
    static constexpr int WAVE_BYTES = TMR * 4 * UNIT;
    static constexpr int REGION = WAVE_BYTES > BM * 128 ? WAVE_BYTES : BM * 128;
    static_assert(TM % ROUNDS == 0, "rounds");

    struct Smem {
        __attribute__((aligned(16))) unsigned char t[KS * REGION];   // a wave's A of one stage, then its partial sums
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
        const unsigned b_voff = (unsigned)((8 * kq * N + 4 * li) * 4), t_voff = (unsigned)((8 * kq * N + G4 * 64 + R * li) * 4);

        shared_with_asm(sm.t);
        f32x4 acc[TM][NB];
        float rb[NB][8];
        // Eight lanes a row, chunk c of row r at c ^ ((r >> 1) & 7): the reads in MFMA layout below then meet no bank twice.
        unsigned a_voff[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) a_voff[h] = (unsigned)(((8 * h + (lane >> 3)) * K + 4 * ((lane & 7) ^ (4 * h + (lane >> 4)))) * 4);
        unsigned char* const region = sm.t + wave * REGION;
        const unsigned char* const a_read = region + li * 128 + ((2 * kq) ^ ((li >> 1) & 6)) * 16;
        const int a_odd = (li >> 1) & 1 ? 16 : 0;
        auto load_a = [&](int s) {
#pragma unroll
            for (int r = 0; r < 2 * TM; ++r)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(ar, (__attribute__((address_space(3))) void*)(region + r * 1024), 16, a_voff[r % 2], s * 128 + r / 2 * 16 * K * 4, 0, 0);
        };
        // 64-column group g, or (g = G4) the 16 R columns past the last one
        auto load_b = [&](int g, int s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int at = (s * 32 + e) * (N * 4);
                if (g < G4) {
                    const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(br, b_voff + g * 256, at, 0));
#pragma unroll
                    for (int c = 0; c < 4; ++c) rb[4 * g + c][e] = v[c];
                } else if constexpr (R == 3) {
                    const auto v = __builtin_amdgcn_raw_buffer_load_b96(br, t_voff, at, 0);
#pragma unroll
                    for (int c = 0; c < 3; ++c) rb[4 * G4 + c][e] = __builtin_bit_cast(float, (unsigned)v[c]);
                } else if constexpr (R == 2) {
                    const auto v = __builtin_amdgcn_raw_buffer_load_b64(br, t_voff, at, 0);
#pragma unroll
                    for (int c = 0; c < 2; ++c) rb[4 * G4 + c][e] = __builtin_bit_cast(float, (unsigned)v[c]);
                } else if constexpr (R == 1) {
                    rb[4 * G4][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, t_voff, at, 0));
                }
            }
        };
        // This wave's loads into LDS have landed: what is on its way after them are `behind` loads, those of B of the same stage.  Its
        // reads of A are done: the loads of the next stage may overwrite it.  (The build looks for the remark in the assembly and
        // counts there, and that nothing is written to LDS while such a load is on its way: the compiler waits for neither.)
        auto a_landed = [&](auto behind) {
#if defined(__HIP_DEVICE_COMPILE__)
            asm volatile("s_waitcnt vmcnt(%0) ; loads into LDS have landed" : : "n"(decltype(behind)::value) : "memory");
#endif
        };
        auto a_read_done = [&]() {
#if defined(__HIP_DEVICE_COMPILE__)
            asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
#endif
            __builtin_amdgcn_sched_barrier(0);
        };
        unsigned pa[TM][3][4], pb[2][4], qb[2][4];          // the parts of A; part 0 of two column blocks of B, parts 1 and 2 of one
        unsigned left = 0;                                  // see split.h
        auto convert_a = [&](int tm) {
            f32x4 ra[2];
            ra[0] = *reinterpret_cast<const f32x4*>(a_read + tm * 2048 + a_odd);
            ra[1] = *reinterpret_cast<const f32x4*>(a_read + tm * 2048 + 16 - a_odd);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                split2(ra[j / 2][2 * (j % 2)], ra[j / 2][2 * (j % 2) + 1], pa[tm][0][j], pa[tm][1][j], pa[tm][2][j], left);
                gather_left(left);
            }
        };
        // part 0 of column block b, and what is left in the place of its values; the other parts
        auto first_b = [&](int b) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const unsigned p = pb[b & 1][j] = pack_bf16(rb[b][2 * j], rb[b][2 * j + 1]);
                rb[b][2 * j] -= __builtin_bit_cast(float, p << 16);
                rb[b][2 * j + 1] -= __builtin_bit_cast(float, p & 0xffff0000u);
            }
        };
        auto others_b = [&](int b) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                split2_left(rb[b][2 * j], rb[b][2 * j + 1], qb[0][j], qb[1][j], left);
                gather_left(left);
            }
        };
        const auto group_of = [](int b) constexpr { return b / 4; };

#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[tm][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        load_a(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < G4 + (R > 0); ++g) load_b(g, 0);
#pragma unroll 1
        for (int s = 0; s < NS; ++s) {
            const int ahead = s + 1 < NS ? s + 1 : s;       // past the end: the last one again (see behind the loop)
            a_landed(std::integral_constant<int, 8 * (G4 + (R > 0))>{});
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) convert_a(tm);
            a_read_done();
            load_a(ahead);
            __builtin_amdgcn_sched_barrier(0);
            first_b(0);
            others_b(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                // Parts 1 and 2 of a block are done with after half its MFMAs: those of the next one take their registers.
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (b + 1 < NB) {
                        if (h == 0) first_b(b + 1);
                        else others_b(b + 1);
                    }
                    // a group's registers are free once its last block has been taken apart
                    if (h == 1 && b + 1 < NB && (b + 2 == NB || group_of(b + 2) != group_of(b + 1))) load_b(group_of(b + 1), ahead);
#pragma unroll
                    for (int t = 3 * h; t < 3 * h + 3; ++t)
#pragma unroll
                        for (int tm = 0; tm < TM; ++tm) {
                            const unsigned(&p)[4] = pa[tm][SplitTerms::A[t]];
                            const unsigned(&q)[4] = SplitTerms::B[t] == 0 ? pb[b & 1] : qb[SplitTerms::B[t] - 1];
                            acc[tm][b] = mfma_bf16(u32x4{p[0], p[1], p[2], p[3]}, u32x4{q[0], q[1], q[2], q[3]}, acc[tm][b]);
                        }
#pragma unroll
                    for (int r = 0; r < 3 * TM; ++r) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                          // an MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, (25 + 3 * TM - 1) / (3 * TM), 0);   // vector instructions
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
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
        // The A that the last stage loaded again lands where the partial sums go.
        a_landed(std::integral_constant<int, 0>{});

        // component v of row block tm (row 4 rg + v of it) is unit 4 tm + v, finished by wave unit % KS
        unsigned char* const part = sm.t + lane * 16;
        unsigned char* const part1 = sm.t + G4 * 1024 + lane * 4 * R;
        auto hand_over = [&](int r, float add) {
#pragma unroll
            for (int tm = 0; tm < TMR; ++tm)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int at = wave * REGION + (tm * 4 + v) * UNIT;
                    const f32x4(&a)[NB] = acc[r * TMR + tm];
#pragma unroll
                    for (int g = 0; g < G4; ++g) *reinterpret_cast<f32x4*>(part + at + g * 1024) = f32x4{a[4 * g][v], a[4 * g + 1][v], a[4 * g + 2][v], a[4 * g + 3][v]} + add;
#pragma unroll
                    for (int g = 0; g < R; ++g) *reinterpret_cast<float*>(part1 + at + g * 4) = a[4 * G4 + g][v] + add;
                }
        };
        constexpr int NU = TMR * 4 / KS;                    // units a wave finishes
        static_assert(TMR * 4 % KS == 0, "every wave finishes as many rows");
        f32x4 o4[NU][G4 > 0 ? G4 : 1];
        float o1[NU][R > 0 ? R : 1];
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
                    for (int w = 1; w < KS; ++w) o += *reinterpret_cast<const f32x4*>(part + w * REGION + u * UNIT + g * 1024);
                    o4[i][g] = o;
                    nan = nan != nan ? nan : o[0];
                }
#pragma unroll
                for (int g = 0; g < R; ++g) {
                    float o = *reinterpret_cast<const float*>(part1 + u * UNIT + g * 4);
#pragma unroll
                    for (int w = 1; w < KS; ++w) o += *reinterpret_cast<const float*>(part1 + w * REGION + u * UNIT + g * 4);
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
                f32x4 nb[2][G4 > 0 ? G4 : 1];
                float nt[2][R > 0 ? R : 1];
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
                        for (int g = 0; g < R; ++g)
                            nt[e][g] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(br, (unsigned)((kq * N + G4 * 64 + R * li + g) * 4), (k + 4 * e) * (N * 4), 0));
                    }
                };
                fetch(0);
#pragma unroll 1
                for (int k = 0; k < KW; k += 8) {
                    float a[2][TM];
                    f32x4 v[2][G4 > 0 ? G4 : 1];
                    float w[2][R > 0 ? R : 1];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
#pragma unroll
                        for (int tm = 0; tm < TM; ++tm) a[e][tm] = na[e][tm];
#pragma unroll
                        for (int g = 0; g < G4; ++g) v[e][g] = nb[e][g];
#pragma unroll
                        for (int g = 0; g < R; ++g) w[e][g] = nt[e][g];
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
                for (int g = 0; g < R; ++g) row[G4 * 64 + R * li + g] = epilogue(o1[i][g]);
            }
        }
    }
};

}  // namespace bfuse
