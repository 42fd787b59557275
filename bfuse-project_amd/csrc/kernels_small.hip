// Small instances of every operator body and fusion form.  They exist for the parity tests:
// shapes the CPU oracle evaluates in full, tile configurations the five headline pairs do
// not reach (single-wave GEMM without LDS reduction, 16-column groups only, deeper
// prefetch, multi-group convolution, several K-steps / M-tiles of the bf16 GEMM), sides with
// different grid sizes under horizontal fusion, and the ratio / proportional block patterns.
#include "fuse.h"
#include "ops_ceiling.h"
#include "ops_conv.h"
#include "ops_conv_1x1.h"
#include "ops_conv_few.h"
#include "ops_conv_rect.h"
#include "ops_conv_split.h"
#include "ops_conv_tile.h"
#include "ops_gemm_bf16.h"
#include "ops_gemm_f32.h"
#include "ops_gemm_f32_dma.h"
#include "ops_gemm_split.h"
#include "ops_gemm_tile.h"
#include "ops_layout.h"
#include "ops_pool.h"
#include "ops_rowwise.h"

using namespace bfuse;

BFUSE_MODULE_PROLOGUE()

// Test operator for the side barrier's give-up path: the two waves of a workgroup swap their
// values through LDS across one barrier, y[g] = x[partner of g] + f[g].  Under a side barrier
// (GroupSync) wave 0 then takes ONE MORE barrier that wave 1 never reaches: the wait is bounded, so
// it gives up, the kernel ends normally with the right output, and the host must report
// BFUSE_ERR_SYNC.  Under the hardware barrier (standalone, block fusion) the body is well formed.
template <int NBLOCKS_, int TAG_>
struct SyncProbe {
    static constexpr int THREADS = 128;
    static constexpr Dims3 GRID{NBLOCKS_, 1, 1};
    static constexpr Dims3 BLOCK{THREADS, 1, 1};
    static constexpr bool HAS_BARRIERS = true;
    struct Smem {
        float v[THREADS];
    };
    template <class Sync>
    __device__ static __forceinline__ void run(int vblock, int tid, Smem& sm, const void* I, const void* F, void* O, Sync sync)
    {
        const int g = vblock * THREADS + tid;
        sm.v[tid] = static_cast<const float*>(I)[g];
        sync();
        static_cast<float*>(O)[g] = sm.v[tid ^ 64] + static_cast<const float*>(F)[g];
        if constexpr (std::is_same<Sync, GroupSync>::value) {
            if (tid < 64) sync();   // unmatched on purpose: bounded wait, then the give-up is recorded
        }
    }
};
using SyncProbeA = SyncProbe<4, 0>;
using SyncProbeB = SyncProbe<6, 1>;

using GemmS1 = GemmF32<64, 48, 32, 16, 48, 1>;                        // one wave, a 32- and a 16-column group
using GemmS2 = GemmF32<96, 192, 128, 32, 64, 2, kEpiGeluTanh, 3>;     // 2 waves, GELU, 3 register stages
using GemmS3 = GemmF32<32, 144, 256, 32, 144, 4>;                     // the 64+64+16 column split, one tile
using GemmS7 = GemmF32<80, 112, 32, 32, 64, 1>;                        // tiles that do not divide the problem: rows 0, 32, 48 and columns 0, 48 (the last tiles overlap their neighbours)
using GemmS8 = GemmF32<48, 80, 64, 32, 64, 2, kEpiNone, 2, 1, true, 3>;   // the same on three batched products with B [N, K] and two waves over K
using GemmS9 = GemmF32<256, 64, 32, 128, 64, 1>;                       // 128 x 64 tiles: 32 accumulator blocks, a kernel of one wave per SIMD (MIN_WAVES_PER_EU), also when fused
using GemmS5 = GemmF32Dma<128, 192, 160, 32, 96, 2>;                  // private LDS rings (GemmF32Ring), two waves split K, ten 8-k stages each
using GemmS6 = GemmF32Dma<64, 288, 192, 32, 144, 4, kEpiGeluTanh>;    // the 32x144 tile on the ring (48 k a wave is no whole stage of GemmSplitK; partial last B load), four waves, GELU
using BiasReluS = BiasRelu<4096, 64, 4>;
using LayerNormS = LayerNorm<8, 256, 2, 1>;
using SoftmaxS = SoftmaxCausal<2, 256, 2, 2, 2>;
using ConvS1 = Conv3x3F32Lds<16, 16, 8, 8, 16, 1, 1>;                 // one channel group, one wave
using ConvS2 = Conv3x3F32Lds<32, 32, 12, 12, 16, 1, 2>;               // two channel groups on two waves
using ConvS3 = Conv3x3F32Lds<64, 16, 8, 16, 16, 2, 2>;                // two groups per wave, two pixel blocks
using PoolS = MaxPool3x3S2<4, 16, 16, 64>;
using Conv1S1 = Conv1x1F32<32, 32, 5, 5, 1, 32, 4, 3>;                 // streamed 1x1: three images of 25 pixels = three ragged tiles in one workgroup, its fourth wave without a tile
using Conv1S2 = Conv1x1F32<96, 48, 9, 9, 1, 16, 2, 5>;                 // 64 + 17 pixels per image, three channel tiles, two filter chunks of 48 channels (192 staging units on 128 threads)
using Conv1S3 = Conv1x1F32<16, 16, 9, 7, 2, 16, 1, 2>;                 // stride 2 (9 x 7 -> 5 x 4), one wave per workgroup: no barrier
using GemmB1 = GemmBf16NTDma<128, 1792, 64, 128, 224, 2>;             // one K-step
using GemmB2 = GemmBf16NTDma<128, 1792, 192, 128, 224, 2>;            // two stages, three K-steps
using GemmB3 = GemmBf16NTDma<256, 1792, 320, 128, 224, 3>;            // two M-tiles, ring of three, five K-steps
using GemmB5 = GemmBf16NTDma<256, 1792, 320, 128, 224, 3, 4, 4, 2>;   // the same with eight waves (uneven load groups per wave)
using GemmB8 = GemmBf16NTDma<256, 1792, 384, 128, 224, 3, 4, 4, 2, 4, 11>;   // eight compute + four producer waves, early barrier, six K-steps (all after the rolled loop)
using GemmB9 = GemmBf16NTDma<256, 1792, 448, 128, 224, 3, 4, 4, 2, 2, 10>;   // eight compute + two producer waves, early barrier, seven K-steps (one round of the rolled loop, then the last step)
using GemmB11 = GemmBf16NTDma<128, 1024, 320, 64, 128, 3, 2, 2, 2, 2, 6>;   // 64 x 128 tiles, four compute waves (2 x 2) of 32 x 64 + two producer waves, read-ahead of two, early barrier
using NormRopeS = RmsNormRope<6, 8, 128, 2>;

BFUSE_KERNEL(gemm_f32_64x32x48, GemmS1, ({{64, 32, 1, 1}, 4}), ({{32, 48, 1, 1}, 4}), ({{64, 48, 1, 1}, 4}))
BFUSE_KERNEL(gemm_gelu_f32_96x128x192, GemmS2, ({{96, 128, 1, 1}, 4}), ({{128, 192, 1, 1}, 4}), ({{96, 192, 1, 1}, 4}))
BFUSE_KERNEL(gemm_f32_32x256x144, GemmS3, ({{32, 256, 1, 1}, 4}), ({{256, 144, 1, 1}, 4}), ({{32, 144, 1, 1}, 4}))
BFUSE_KERNEL(gemm_f32_80x32x112, GemmS7, ({{80, 32, 1, 1}, 4}), ({{32, 112, 1, 1}, 4}), ({{80, 112, 1, 1}, 4}))
BFUSE_KERNEL(bgemm_f32_3x48x64x80, GemmS8, ({{3, 48, 64, 1}, 4}), ({{3, 80, 64, 1}, 4}), ({{3, 48, 80, 1}, 4}))
BFUSE_KERNEL(gemm_f32_256x32x64_t128, GemmS9, ({{256, 32, 1, 1}, 4}), ({{32, 64, 1, 1}, 4}), ({{256, 64, 1, 1}, 4}))
BFUSE_KERNEL(gemm_f32_128x160x192_d, GemmS5, ({{128, 160, 1, 1}, 4}), ({{160, 192, 1, 1}, 4}), ({{128, 192, 1, 1}, 4}))
BFUSE_KERNEL(gemm_gelu_f32_64x192x288_d, GemmS6, ({{64, 192, 1, 1}, 4}), ({{192, 288, 1, 1}, 4}), ({{64, 288, 1, 1}, 4}))
BFUSE_KERNEL(bias_relu_4096, BiasReluS, ({{4096, 1, 1, 1}, 4}), ({{4096, 1, 1, 1}, 4}), ({{4096, 1, 1, 1}, 4}))
BFUSE_KERNEL(layernorm_8x256, LayerNormS, ({{8, 256, 1, 1}, 4}), ({{2, 256, 1, 1}, 4}), ({{8, 256, 1, 1}, 4}))
BFUSE_KERNEL(softmax_causal_2x256x256, SoftmaxS, ({{2, 256, 256, 1}, 4}), ({{1, 1, 1, 1}, 4}), ({{2, 256, 256, 1}, 4}))
BFUSE_KERNEL(conv3x3_f32_16x8x8_16, ConvS1, ({{1, 16, 8, 8}, 4}), ({{16, 16, 3, 3}, 4}), ({{1, 16, 8, 8}, 4}))
BFUSE_KERNEL(conv3x3_f32_32x12x12_32, ConvS2, ({{1, 32, 12, 12}, 4}), ({{32, 32, 3, 3}, 4}), ({{1, 32, 12, 12}, 4}))
BFUSE_KERNEL(conv3x3_f32_64x8x16_16, ConvS3, ({{1, 64, 8, 16}, 4}), ({{16, 64, 3, 3}, 4}), ({{1, 16, 8, 16}, 4}))
BFUSE_KERNEL(conv1x1s1p0_f32_3x32x5x5_32, Conv1S1, ({{3, 32, 5, 5}, 4}), ({{32, 32, 1, 1}, 4}), ({{3, 32, 5, 5}, 4}))
BFUSE_KERNEL(conv1x1s1p0_f32_5x96x9x9_48, Conv1S2, ({{5, 96, 9, 9}, 4}), ({{48, 96, 1, 1}, 4}), ({{5, 48, 9, 9}, 4}))
BFUSE_KERNEL(conv1x1s2p0_f32_2x16x9x7_16, Conv1S3, ({{2, 16, 9, 7}, 4}), ({{16, 16, 1, 1}, 4}), ({{2, 16, 5, 4}, 4}))
BFUSE_KERNEL(maxpool3x3s2_f32_4x16x16, PoolS, ({{1, 4, 16, 16}, 4}), ({{1, 1, 1, 1}, 4}), ({{1, 4, 8, 8}, 4}))
BFUSE_KERNEL(gemm_bf16_128x64x1792, GemmB1, ({{128, 64, 1, 1}, 2}), ({{1792, 64, 1, 1}, 2}), ({{128, 1792, 1, 1}, 2}))
BFUSE_KERNEL(gemm_bf16_128x192x1792, GemmB2, ({{128, 192, 1, 1}, 2}), ({{1792, 192, 1, 1}, 2}), ({{128, 1792, 1, 1}, 2}))
BFUSE_KERNEL(gemm_bf16_256x320x1792, GemmB3, ({{256, 320, 1, 1}, 2}), ({{1792, 320, 1, 1}, 2}), ({{256, 1792, 1, 1}, 2}))
BFUSE_KERNEL(gemm_bf16_256x320x1792_w8, GemmB5, ({{256, 320, 1, 1}, 2}), ({{1792, 320, 1, 1}, 2}), ({{256, 1792, 1, 1}, 2}))
BFUSE_KERNEL(gemm_bf16_256x384x1792_p, GemmB8, ({{256, 384, 1, 1}, 2}), ({{1792, 384, 1, 1}, 2}), ({{256, 1792, 1, 1}, 2}))
BFUSE_KERNEL(gemm_bf16_256x448x1792_p2, GemmB9, ({{256, 448, 1, 1}, 2}), ({{1792, 448, 1, 1}, 2}), ({{256, 1792, 1, 1}, 2}))
BFUSE_KERNEL(gemm_bf16_128x320x1024_t64, GemmB11, ({{128, 320, 1, 1}, 2}), ({{1024, 320, 1, 1}, 2}), ({{128, 1024, 1, 1}, 2}))
BFUSE_KERNEL(rmsnorm_rope_bf16_6x1024, NormRopeS, ({{6, 1024, 1, 1}, 2}), ({{(int)NormRopeS::F_BYTES, 1, 1, 1}, 1}), ({{6, 1024, 1, 1}, 2}))

// [128, 192] -> [192, 128], 16-bit elements: 2 x 3 tiles
using TransposeS = Transpose16<128, 192>;
BFUSE_KERNEL(transpose16_128x192, TransposeS, ({{128, 192, 1, 1}, 2}), ({{1, 1, 1, 1}, 2}), ({{192, 128, 1, 1}, 2}))

// calibration kernel for the memory counters: 64 MiB read, 64 MiB written
using Copy64M = CopyF32<16777216, 256>;
BFUSE_KERNEL(copy_f32_16777216, Copy64M, ({{16777216, 1, 1, 1}, 4}), ({{1, 1, 1, 1}, 4}), ({{16777216, 1, 1, 1}, 4}))

// what the matrix cores sustain with nothing else going on: 2000 (bf16) / 1000 (fp32) rounds of 14
// independent MFMAs per wave, 0.94 TFLOP / 0.059 TFLOP per launch (about 0.6 / 0.4 ms)
using MfmaStreamBf16 = MfmaStream<true, 2000>;
using MfmaStreamF32 = MfmaStream<false, 1000>;
BFUSE_KERNEL(mfma_stream_bf16_2000, MfmaStreamBf16, ({{1, 1, 1, 1}, 4}), ({{1, 1, 1, 1}, 4}), ({{256, 512, 1, 1}, 4}))
BFUSE_KERNEL(mfma_stream_f32_1000, MfmaStreamF32, ({{1, 1, 1, 1}, 4}), ({{1, 1, 1, 1}, 4}), ({{256, 512, 1, 1}, 4}))

// horizontal fusion with unequal grids (9 GEMM tiles, 4 element-wise blocks) and a barrier side
BFUSE_HFUSE_KERNEL(gemm_gelu_f32_96x128x192, GemmS2, bias_relu_4096, BiasReluS)
// both sides carry a barrier: two LDS-counter barriers in one workgroup
BFUSE_HFUSE_KERNEL(gemm_gelu_f32_96x128x192, GemmS2, conv3x3_f32_32x12x12_32, ConvS2)
// ratio 2:1 zig-zag (18 conv tiles, 9 GEMM tiles), proportional, chunked with a remainder
BFUSE_BFUSE_KERNEL(conv3x3_f32_32x12x12_32, ConvS2, gemm_gelu_f32_96x128x192, GemmS2, , bfuse::kZigzag, 2, 1)
BFUSE_BFUSE_KERNEL(conv3x3_f32_32x12x12_32, ConvS2, gemm_gelu_f32_96x128x192, GemmS2, _p1, bfuse::kProportional, 1, 1)
BFUSE_BFUSE_KERNEL(conv3x3_f32_32x12x12_32, ConvS2, gemm_gelu_f32_96x128x192, GemmS2, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(layernorm_8x256, LayerNormS, softmax_causal_2x256x256, SoftmaxS, , bfuse::kZigzag, 1, 1)
BFUSE_BFUSE_KERNEL(gemm_bf16_256x320x1792, GemmB3, rmsnorm_rope_bf16_6x1024, NormRopeS, _c8, bfuse::kChunked, 8, 1)
BFUSE_HFUSE_KERNEL(maxpool3x3s2_f32_4x16x16, PoolS, layernorm_8x256, LayerNormS)
// a side with a barrier in its K loop under horizontal fusion, both sides synchronising: its fence-free
// barriers become the LDS-counter one
BFUSE_HFUSE_KERNEL(gemm_bf16_256x320x1792_w8, GemmB5, gemm_f32_128x160x192_d, GemmS5)
// (the producer-wave GEMMs are not paired with a synchronising partner: their K loop under the LDS-counter
// barrier needs more scalar registers than there are, and the build refuses kernels that spill)
// the same GEMM with producer waves keeps the hardware barrier in its K loop and the norm waves join
// its first four barriers (16 GEMM tiles, 3 norm workgroups: most workgroups have no norm waves at all)
BFUSE_HFUSE_KERNEL(gemm_bf16_256x384x1792_p, GemmB8, rmsnorm_rope_bf16_6x1024, NormRopeS)
BFUSE_HFUSE_KERNEL(gemm_bf16_256x448x1792_p2, GemmB9, rmsnorm_rope_bf16_6x1024, NormRopeS)
// run-time plans / persistent workgroups: equal and unequal workgroup widths, barrier-bearing sides
BFUSE_BFUSE_RT_KERNEL(conv3x3_f32_32x12x12_32, ConvS2, gemm_gelu_f32_96x128x192, GemmS2)
BFUSE_BFUSE_RT_KERNEL(layernorm_8x256, LayerNormS, softmax_causal_2x256x256, SoftmaxS)
BFUSE_BFUSE_RT_KERNEL(gemm_bf16_256x320x1792_w8, GemmB5, rmsnorm_rope_bf16_6x1024, NormRopeS)
BFUSE_BFUSE_RT_KERNEL(gemm_f32_128x160x192_d, GemmS5, bias_relu_4096, BiasReluS)
BFUSE_HFUSE_KERNEL(gemm_f32_128x160x192_d, GemmS5, bias_relu_4096, BiasReluS)
BFUSE_BFUSE_KERNEL(gemm_gelu_f32_64x192x288_d, GemmS6, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_HFUSE_KERNEL(conv3x3_f32_32x12x12_32, ConvS2, bias_relu_4096, BiasReluS)
BFUSE_BFUSE_KERNEL(conv3x3_f32_64x8x16_16, ConvS3, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
// both sides synchronise (each split-K GEMM's reduction barriers): each side gets LDS arrival counters of its own
BFUSE_HFUSE_KERNEL(gemm_f32_128x160x192_d, GemmS5, gemm_gelu_f32_64x192x288_d, GemmS6)
// the streamed 1x1 convolution (a barrier per filter chunk): block-fused, thread-fused with a side that never
// synchronises, and with one that does
BFUSE_BFUSE_KERNEL(conv1x1s1p0_f32_3x32x5x5_32, Conv1S1, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_HFUSE_KERNEL(conv1x1s1p0_f32_5x96x9x9_48, Conv1S2, bias_relu_4096, BiasReluS)
BFUSE_HFUSE_KERNEL(conv1x1s1p0_f32_5x96x9x9_48, Conv1S2, conv3x3_f32_32x12x12_32, ConvS2)
BFUSE_BFUSE_KERNEL(conv1x1s2p0_f32_2x16x9x7_16, Conv1S3, bias_relu_4096, BiasReluS, , bfuse::kZigzag, 1, 1)
// a side that needs more than the 256 registers of two waves per SIMD: the fused kernels are compiled for one
static_assert(bfuse::min_waves<GemmS9>() == 1 && bfuse::min_waves<GemmS9, BiasReluS>() == 1 && bfuse::min_waves<GemmS1, BiasReluS>() == bfuse::kMinWavesPerEu,
              "a fused kernel takes the smallest wave count of its sides");
BFUSE_BFUSE_KERNEL(gemm_f32_256x32x64_t128, GemmS9, bias_relu_4096, BiasReluS, , bfuse::kZigzag, 1, 1)
BFUSE_HFUSE_KERNEL(gemm_f32_256x32x64_t128, GemmS9, bias_relu_4096, BiasReluS)
// overlapping last tiles: the shared elements are written twice with the same bits, also inside fused kernels
BFUSE_BFUSE_KERNEL(gemm_f32_80x32x112, GemmS7, layernorm_8x256, LayerNormS, , bfuse::kZigzag, 1, 1)
BFUSE_HFUSE_KERNEL(bgemm_f32_3x48x64x80, GemmS8, bias_relu_4096, BiasReluS)
// the give-up path of the side barrier, forced from the host with a small spin limit
BFUSE_KERNEL(selftest_sync_a, SyncProbeA, ({{512, 1, 1, 1}, 4}), ({{512, 1, 1, 1}, 4}), ({{512, 1, 1, 1}, 4}))
BFUSE_KERNEL(selftest_sync_b, SyncProbeB, ({{768, 1, 1, 1}, 4}), ({{768, 1, 1, 1}, 4}), ({{768, 1, 1, 1}, 4}))
BFUSE_HFUSE_KERNEL(selftest_sync_a, SyncProbeA, selftest_sync_b, SyncProbeB)

// The shared-tile convolution at the edges of its tiles (found by name only, so that nothing that walks the registry meets
// them): tiles that run over several images, last tiles past the batch, strides, even and large filters, few stages and
// many.  <CI, CO, H, W, KH, KW, S, P, BM, 16-pixel blocks, images, waves over BM>
#define CONV_TILE_TEST(TAG, CI, CO, H, W, KH, KW, S, P, BM, PB, N, WM)                                             \
    using ConvT_##TAG = ConvF32Lds<CI, CO, H, W, KH, KW, S, P, BM, PB, 4, N, WM>;                                  \
    BFUSE_KERNEL(selftest_conv_tile_##TAG, ConvT_##TAG, ({{N, CI, H, W}, 4}), ({{CO, CI, KH, KW}, 4}),             \
                 ({{N, CO, (H - KH + 2 * P) / S + 1, (W - KW + 2 * P) / S + 1}, 4}))
CONV_TILE_TEST(a, 16, 32, 5, 5, 3, 3, 1, 1, 32, 4, 3, 1)         // 75 pixels of three images in two tiles of 64
CONV_TILE_TEST(b, 32, 64, 9, 7, 3, 3, 2, 0, 32, 4, 5, 2)         // stride 2, 60 pixels of five images in one tile
CONV_TILE_TEST(c, 16, 16, 11, 6, 5, 5, 1, 2, 16, 8, 4, 1)        // 5 x 5, tiles of 128 over images of 66
CONV_TILE_TEST(d, 16, 64, 20, 13, 3, 3, 4, 1, 64, 4, 9, 2)       // stride 4, one window row per four image rows
CONV_TILE_TEST(e, 48, 96, 8, 33, 3, 1, 1, 1, 96, 8, 7, 2)        // 3 x 1 filter: an odd number of columns, twelve stages
CONV_TILE_TEST(f, 16, 128, 7, 7, 3, 3, 1, 1, 128, 10, 5, 2)      // 245 pixels in two tiles of 160, five blocks a wave
CONV_TILE_TEST(g, 20, 48, 11, 11, 3, 3, 1, 1, 48, 20, 3, 1)      // 363 pixels in two tiles of 320, an odd number of stages
CONV_TILE_TEST(h, 64, 32, 9, 9, 3, 3, 1, 1, 32, 4, 3, 1)         // sixteen stages, summed three at a time
BFUSE_HFUSE_KERNEL(selftest_conv_tile_a, ConvT_a, bias_relu_4096, BiasReluS)
BFUSE_BFUSE_KERNEL(selftest_conv_tile_b, ConvT_b, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_HFUSE_KERNEL(selftest_conv_tile_c, ConvT_c, conv3x3_f32_32x12x12_32, ConvS2)

// The per-wave convolutions at the edges of what they stage (found by name only): image rows that end or begin inside a vector, rows of
// one, two and four floats a load, filters that come through LDS at once and one row block after the other, those that do not (more than nine taps), groups
// that follow each other in a wave's tile.
#define CONV_STAGED_TEST(TAG, N, CI, H, W, CO, KH, KW, S, P, ...)                                                  \
    using ConvW_##TAG = __VA_ARGS__;                                                                               \
    BFUSE_KERNEL(selftest_conv_staged_##TAG, ConvW_##TAG, ({{N, CI, H, W}, 4}), ({{CO, CI, KH, KW}, 4}),           \
                 ({{N, CO, (H - KH + 2 * P) / S + 1, (W - KW + 2 * P) / S + 1}, 4}))
CONV_STAGED_TEST(a, 2, 3, 21, 37, 16, 5, 5, 1, 2, ConvF32Few<3, 16, 21, 37, 5, 5, 1, 2, 16, 2, 1, 2>)             // a vector begins two floats before the row
CONV_STAGED_TEST(b, 2, 16, 19, 50, 32, 3, 3, 1, 1, ConvF32Rect<16, 32, 19, 50, 3, 3, 1, 1, 32, 4, 1, 2>)          // one float before, two row blocks
CONV_STAGED_TEST(c, 3, 4, 23, 35, 32, 3, 3, 2, 1, ConvF32Few<4, 32, 23, 35, 3, 3, 2, 1, 32, 2, 1, 3>)            // four channels, two row blocks
CONV_STAGED_TEST(d, 1, 2, 30, 30, 16, 11, 11, 1, 5, ConvF32Few<2, 16, 30, 30, 11, 11, 1, 5, 16, 1, 1, 1>)        // 121 taps; the second vector begins before the row
CONV_STAGED_TEST(e, 2, 64, 18, 41, 16, 3, 3, 1, 0, ConvF32Rect<64, 16, 18, 41, 3, 3, 1, 0, 16, 4, 2, 2>)          // two waves of two groups, no padding
CONV_STAGED_TEST(f, 1, 3, 29, 62, 16, 7, 7, 2, 3, ConvF32Few<3, 16, 29, 62, 7, 7, 2, 3, 16, 4, 1, 1>)            // 9408 bytes of filters, three floats before the row
CONV_STAGED_TEST(g, 1, 32, 9, 10, 32, 3, 3, 1, 1, ConvF32Lds<32, 32, 9, 10, 3, 3, 1, 1, 32, 2, 1, 1>)             // 8-byte loads, two groups, two row blocks
CONV_STAGED_TEST(h, 1, 48, 7, 7, 16, 3, 3, 2, 1, ConvF32Lds<48, 16, 7, 7, 3, 3, 2, 1, 16, 1, 3, 1>)               // 4-byte loads, three waves
CONV_STAGED_TEST(i, 3, 16, 13, 11, 16, 5, 5, 1, 2, ConvF32Lds<16, 16, 13, 11, 5, 5, 1, 2, 16, 4, 1, 3>)           // 25 taps, rows as one span
CONV_STAGED_TEST(j, 3, 32, 15, 13, 16, 3, 3, 1, 1, ConvF32Lds<32, 16, 15, 13, 3, 3, 1, 1, 16, 4, 1, 3>)           // the same, two groups, filters through LDS
CONV_STAGED_TEST(k, 2, 16, 10, 12, 16, 1, 3, 1, 1, ConvF32Lds<16, 16, 10, 12, 1, 3, 1, 1, 16, 4, 1, 2>)           // three taps
CONV_STAGED_TEST(l, 1, 32, 8, 12, 32, 3, 3, 1, 1, Conv3x3F32Lds<32, 32, 8, 12, 32, 2, 1>)                        // two groups, two row blocks
CONV_STAGED_TEST(m, 2, 3, 11, 131, 32, 3, 3, 1, 0, ConvF32Few<3, 32, 11, 131, 3, 3, 1, 0, 32, 2, 4, 2>)            // four columns a lane, 129 of 192: a quad cut after one
CONV_STAGED_TEST(n, 2, 1, 13, 150, 16, 5, 5, 2, 2, ConvF32Few<1, 16, 13, 150, 5, 5, 2, 2, 16, 2, 4, 2>)            // one channel: a row a lane group and five taps of one that is left; cut after three
CONV_STAGED_TEST(o, 2, 2, 12, 80, 32, 3, 3, 1, 1, ConvF32Few<2, 32, 12, 80, 3, 3, 1, 1, 32, 2, 4, 2, true>)        // two rows left, six taps; written past the caches
CONV_STAGED_TEST(p, 1, 3, 40, 66, 16, 7, 7, 2, 3, ConvF32Few<3, 16, 40, 66, 7, 7, 2, 3, 16, 8, 1, 1>)              // eight rows
CONV_STAGED_TEST(q, 2, 4, 20, 64, 16, 14, 14, 1, 7, ConvF32Auto<4, 16, 20, 64, 14, 14, 1, 7, 2>)                   // filters that take most of the registers
CONV_STAGED_TEST(r, 2, 4, 18, 64, 16, 13, 13, 1, 6, ConvF32Auto<4, 16, 18, 64, 13, 13, 1, 6, 2>)
CONV_STAGED_TEST(s, 3, 2, 16, 66, 32, 6, 6, 1, 3, ConvF32Auto<2, 32, 16, 66, 6, 6, 1, 3, 3>)                       // half a channel's rows a lane group
// Padding that is wider than a tile: a second and a third tile of a row begin before column 0, inside another vector of theirs.
CONV_STAGED_TEST(x, 2, 16, 7, 62, 16, 3, 3, 1, 17, ConvF32Rect<16, 16, 7, 62, 3, 3, 1, 17, 16, 2, 1, 2>)
CONV_STAGED_TEST(y, 1, 16, 5, 70, 32, 3, 3, 1, 35, ConvF32Rect<16, 32, 5, 70, 3, 3, 1, 35, 32, 4, 1, 1>)
CONV_STAGED_TEST(z, 2, 3, 9, 61, 16, 3, 3, 1, 18, ConvF32Few<3, 16, 9, 61, 3, 3, 1, 18, 16, 4, 1, 2>)
CONV_STAGED_TEST(aa, 1, 4, 12, 64, 32, 3, 3, 1, 67, ConvF32Few<4, 32, 12, 64, 3, 3, 1, 67, 32, 2, 4, 1>)
// Eight loads under way at a time beside many taps: three channels at stride 4 (23 loads), rows that are not whole vectors.
CONV_STAGED_TEST(ca, 1, 3, 30, 190, 16, 13, 13, 4, 6, ConvF32Auto<3, 16, 30, 190, 13, 13, 4, 6, 1>)
CONV_STAGED_TEST(cb, 2, 2, 19, 50, 16, 14, 14, 1, 0, ConvF32Auto<2, 16, 19, 50, 14, 14, 1, 0, 2>)
static_assert(ConvW_ca::Units::JB == 8 && !ConvW_ca::Units::WHOLE && ConvW_cb::MOST == 8);
// Forms of fewer registers beside ten waves: channels and rows one part after the other, fewer loads under way.
CONV_STAGED_TEST(da, 2, 3, 11, 131, 32, 3, 3, 1, 0, LdsReserve<ConvF32Few<3, 32, 11, 131, 3, 3, 1, 0, 32, 2, 4, 2>, 1024>)
CONV_STAGED_TEST(db, 2, 3, 23, 70, 16, 8, 8, 1, 4, ConvF32Auto<3, 16, 23, 70, 8, 8, 1, 4, 2>)                     // eight rows in two parts
CONV_STAGED_TEST(dc, 1, 4, 31, 188, 16, 9, 9, 3, 4, ConvF32Auto<4, 16, 31, 188, 9, 9, 3, 4, 1>)                   // four rows, one at a time
CONV_STAGED_TEST(dd, 1, 32, 14, 22, 16, 3, 3, 1, 1, ConvF32Lds<32, 16, 14, 22, 3, 3, 1, 1, 16, 4, 1, 1>)          // four of the loads that one batch was
BFUSE_BFUSE_KERNEL(selftest_conv_staged_da, Slim<ConvW_da>, gemm_bf16_256x448x1792_p2, GemmB9, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_conv_staged_db, Slim<ConvW_db>, gemm_bf16_256x448x1792_p2, GemmB9, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_conv_staged_dc, Slim<ConvW_dc>, gemm_bf16_256x448x1792_p2, GemmB9, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_conv_staged_dd, Slim<ConvW_dd>, gemm_bf16_256x448x1792_p2, GemmB9, _c4, bfuse::kChunked, 4, 1)
static_assert(Slim<ConvW_da>::TMP == 1 && Slim<ConvW_db>::THP == 4 && ConvW_db::TH == 8 && Slim<ConvW_dc>::THP == 1 && ConvW_dc::TH == 4 && Slim<ConvW_dd>::MOST == 4);
// Images too large for a buffer: their loads on small ones, then 2 GiB of 16 channels and of four (the last floats lie beyond 2^31 bytes; results 16 or 64 times fewer).
template <> inline constexpr bool bfuse::kFarPatch<16 * 11 * 77> = true;
template <> inline constexpr bool bfuse::kFarPatch<3 * 13 * 83> = true;
template <> inline constexpr bool bfuse::kFarPatch<16 * 9 * 15> = true;
template <> inline constexpr bool bfuse::kFarPatch<16 * 10 * 14> = true;
template <> inline constexpr bool bfuse::kFarPatch<16 * 8 * 20> = true;
CONV_STAGED_TEST(ba, 2, 32, 11, 77, 32, 3, 3, 1, 2, ConvF32Rect<32, 32, 11, 77, 3, 3, 1, 2, 32, 4, 2, 2>)
CONV_STAGED_TEST(bb, 2, 3, 13, 83, 16, 5, 5, 1, 2, ConvF32Few<3, 16, 13, 83, 5, 5, 1, 2, 16, 2, 1, 2>)
CONV_STAGED_TEST(bc, 1, 32, 9, 15, 16, 3, 3, 1, 1, ConvF32Lds<32, 16, 9, 15, 3, 3, 1, 1, 16, 2, 1, 1>)
CONV_STAGED_TEST(bd, 1, 16, 10, 14, 16, 5, 3, 2, 1, ConvF32Lds<16, 16, 10, 14, 5, 3, 2, 1, 16, 2, 1, 1>)
CONV_STAGED_TEST(be, 1, 32, 8, 20, 32, 3, 3, 1, 1, Conv3x3F32Lds<32, 32, 8, 20, 32, 2, 2>)
CONV_STAGED_TEST(huge_a, 1, 16, 8192, 4100, 16, 5, 5, 4, 2, ConvF32Auto<16, 16, 8192, 4100, 5, 5, 4, 2, 1>)
CONV_STAGED_TEST(huge_b, 1, 4, 11600, 11601, 16, 8, 8, 8, 1, ConvF32Auto<4, 16, 11600, 11601, 8, 8, 8, 1, 1>)
CONV_STAGED_TEST(huge_c, 1, 16, 1048580, 36, 16, 3, 3, 4, 1, ConvF32Auto<16, 16, 1048580, 36, 3, 3, 4, 1, 1>)
static_assert(ConvTiling<16, 16, 8192, 4100, 5, 5, 4, 2, 1>::RECT && ConvW_huge_a::Source::FAR && ConvW_huge_b::Source::FAR && ConvTiling<4, 16, 11600, 11601, 8, 8, 8, 1, 1>::FEW);
static_assert(!ConvTiling<16, 16, 1048580, 36, 3, 3, 4, 1, 1>::RECT && ConvW_huge_c::Source::FAR && ConvW_ba::Source::FAR && ConvW_be::Source::FAR && !ConvW_x::Source::FAR);
// More loads than are under way at a time, the last batch of them shorter than the others though every lane has a unit in each (25 loads, 16 at a time).
CONV_STAGED_TEST(t, 2, 32, 15, 170, 16, 5, 5, 5, 0, ConvF32Rect<32, 16, 15, 170, 5, 5, 5, 0, 16, 1, 2, 2>)         // a second wave's tile behind the patch
CONV_STAGED_TEST(u, 1, 32, 15, 165, 16, 5, 5, 5, 2, ConvF32Rect<32, 16, 15, 165, 5, 5, 5, 2, 16, 1, 1, 1>)         // a partner's behind it, and a second group's; unrolled
CONV_STAGED_TEST(v, 2, 3, 40, 264, 16, 8, 8, 8, 0, ConvF32Few<3, 16, 40, 264, 8, 8, 8, 0, 16, 2, 1, 2>)            // 24 loads, 16 at a time
CONV_STAGED_TEST(w, 2, 3, 21, 281, 32, 4, 4, 4, 1, ConvF32Few<3, 32, 21, 281, 4, 4, 4, 1, 32, 2, 4, 2>)             // the same with four columns a lane, 70 of 128
BFUSE_HFUSE_KERNEL(selftest_conv_staged_v, ConvW_v, conv3x3_f32_32x12x12_32, ConvS2)
BFUSE_HFUSE_KERNEL(selftest_conv_staged_t, ConvW_t, bias_relu_4096, BiasReluS)
BFUSE_HFUSE_KERNEL(selftest_conv_staged_u, ConvW_u, conv3x3_f32_32x12x12_32, ConvS2)
BFUSE_HFUSE_KERNEL(selftest_conv_staged_m, ConvW_m, bias_relu_4096, BiasReluS)
BFUSE_HFUSE_KERNEL(selftest_conv_staged_a, ConvW_a, bias_relu_4096, BiasReluS)
BFUSE_BFUSE_KERNEL(selftest_conv_staged_g, ConvW_g, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_HFUSE_KERNEL(selftest_conv_staged_l, ConvW_l, bias_relu_4096, BiasReluS)

// The dense product's long stages (16 k): an odd number of them, two waves over K.
using GemmLong = GemmF32Dma<64, 96, 1056, 32, 48, 2>;
static_assert(GemmLong::STAGE == 16);
BFUSE_KERNEL(selftest_gemm_long, GemmLong, ({{64, 1056, 1, 1}, 4}), ({{1056, 96, 1, 1}, 4}), ({{64, 96, 1, 1}, 4}))
BFUSE_HFUSE_KERNEL(selftest_gemm_long, GemmLong, bias_relu_4096, BiasReluS)

// The bf16 product's ring of four stages: eleven K-steps, eight of them in the rolled loop.
using GemmRing4 = GemmBf16NTDma<128, 1024, 704, 64, 128, 4, 2, 2, 2, 2, 6>;
BFUSE_KERNEL(selftest_gemm_ring4, GemmRing4, ({{128, 704, 1, 1}, 2}), ({{1024, 704, 1, 1}, 2}), ({{128, 1024, 1, 1}, 2}))

// The shared-tile product likewise: pixels of images that are no whole chunks, tiles over several images and past the batch,
// strides, row and column tiles that overlap, fewer stages than buffers.
// <M, K, H, W, S, images or products, BM, BN, waves over BM, k per stage, layout, buffers>
#define CONV1_TILE_TEST(TAG, CI, CO, H, W, S, N, BM, BN, WM, KS, NBUF)                                              \
    using GemmT_##TAG = SwapOperands<GemmTile<CO, CI, H, W, S, N, BM, BN, WM, KS, kPix, NBUF>>;                     \
    BFUSE_KERNEL(selftest_gemm_tile_##TAG, GemmT_##TAG, ({{N, CI, H, W}, 4}), ({{CO, CI, 1, 1}, 4}), ({{N, CO, (H - 1) / S + 1, (W - 1) / S + 1}, 4}))
#define BGEMM_TILE_TEST(TAG, B, M, K, N, BM, BN, WM, KS, NBUF)                                                     \
    using GemmT_##TAG = GemmTile<M, K, 1, N, 1, B, BM, BN, WM, KS, kRows, NBUF>;                                   \
    BFUSE_KERNEL(selftest_gemm_tile_##TAG, GemmT_##TAG, ({{B, M, K, 1}, 4}), ({{B, N, K, 1}, 4}), ({{B, M, N, 1}, 4}))
CONV1_TILE_TEST(a, 16, 32, 5, 5, 1, 3, 32, 256, 1, 16, 3)        // one stage, three images of 25 pixels in one tile
CONV1_TILE_TEST(b, 64, 80, 9, 9, 1, 5, 80, 256, 1, 32, 2)        // five images of 81 in two tiles, a row tile that is no whole round of loads
CONV1_TILE_TEST(c, 48, 112, 9, 7, 2, 11, 96, 128, 2, 16, 3)      // stride 2 (20 pixels an image), row tiles that overlap
CONV1_TILE_TEST(d, 32, 64, 8, 8, 1, 7, 64, 128, 2, 16, 3)        // fewer stages than buffers, whole chunks
BGEMM_TILE_TEST(e, 3, 160, 48, 144, 128, 128, 2, 16, 3)          // row and column tiles that overlap
BGEMM_TILE_TEST(f, 8, 64, 32, 64, 64, 64, 4, 32, 2)              // one stage, products dealt to the XCDs
BGEMM_TILE_TEST(g, 2, 64, 512, 64, 64, 64, 4, 32, 3)             // two sums of 256 k
BFUSE_HFUSE_KERNEL(selftest_gemm_tile_c, GemmT_c, bias_relu_4096, BiasReluS)
BFUSE_BFUSE_KERNEL(selftest_gemm_tile_e, GemmT_e, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)

// The product on the bf16 matrix cores: row tiles that overlap and columns past the end, odd and even numbers of stages, threads
// that do a unit twice, a last stage of 8, 16 and 24 k, waves over the columns, groups of waves over K, images and strides.
// <M, K, H, W, S, images or products, 16-row blocks of a wave, waves over rows, over columns, over K, columns, layout>
#define DENSE_SPLIT_TEST(TAG, M, K, N, ...)                                                                        \
    using GemmSp_##TAG = GemmSplit<M, K, 1, N, 1, 1, __VA_ARGS__, kPix>;                                             \
    BFUSE_KERNEL(selftest_gemm_split_##TAG, GemmSp_##TAG, ({{M, K, 1, 1}, 4}), ({{K, N, 1, 1}, 4}), ({{M, N, 1, 1}, 4}))
#define BGEMM_SPLIT_TEST(TAG, B, M, K, N, ...)                                                                     \
    using GemmSp_##TAG = GemmSplit<M, K, 1, N, 1, B, __VA_ARGS__, kRows>;                                            \
    BFUSE_KERNEL(selftest_gemm_split_##TAG, GemmSp_##TAG, ({{B, M, K, 1}, 4}), ({{B, N, K, 1}, 4}), ({{B, M, N, 1}, 4}))
#define CONV1_SPLIT_TEST(TAG, CI, CO, H, W, S, N, ...)                                                             \
    using GemmSp_##TAG = SwapOperands<GemmSplit<CO, CI, H, W, S, N, __VA_ARGS__, kPix>>;                             \
    BFUSE_KERNEL(selftest_gemm_split_##TAG, GemmSp_##TAG, ({{N, CI, H, W}, 4}), ({{CO, CI, 1, 1}, 4}), ({{N, CO, (H - 1) / S + 1, (W - 1) / S + 1}, 4}))
// ... and convolutions: padding, strides, images of odd pixels, a last stage that runs past the window, 30 taps, even filters.
#define CONV_SPLIT_TEST(TAG, CI, CO, H, W, KH, KW, S, P, N, ...)                                                    \
    using GemmSp_##TAG = SwapOperands<GemmSplit<CO, CI * KH * KW, H, W, S, N, __VA_ARGS__, kPix, KH, KW, P>>;          \
    BFUSE_KERNEL(selftest_gemm_split_##TAG, GemmSp_##TAG, ({{N, CI, H, W}, 4}), ({{CO, CI, KH, KW}, 4}),             \
                 ({{N, CO, (H - KH + 2 * P) / S + 1, (W - KW + 2 * P) / S + 1}, 4}))
CONV_SPLIT_TEST(i, 16, 64, 9, 7, 3, 3, 1, 1, 5, 2, 2, 1, 1, 64)
CONV_SPLIT_TEST(j, 24, 48, 17, 17, 3, 3, 2, 0, 3, 1, 3, 1, 1, 128)
CONV_SPLIT_TEST(k, 48, 32, 8, 12, 5, 5, 1, 2, 2, 1, 2, 2, 2, 64)
CONV_SPLIT_TEST(l, 16, 80, 12, 10, 5, 6, 3, 2, 7, 1, 4, 1, 1, 64)
DENSE_SPLIT_TEST(a, 160, 96, 144, 2, 4, 1, 1, 64)
DENSE_SPLIT_TEST(b, 128, 256, 96, 2, 4, 1, 2, 96)
DENSE_SPLIT_TEST(c, 256, 64, 224, 2, 8, 1, 1, 112)
DENSE_SPLIT_TEST(d, 64, 4096, 64, 2, 2, 1, 1, 64)
BGEMM_SPLIT_TEST(e, 8, 64, 72, 80, 1, 2, 2, 1, 64)
BGEMM_SPLIT_TEST(f, 3, 208, 208, 112, 1, 7, 1, 1, 112)
DENSE_SPLIT_TEST(m, 64, 256, 144, 2, 2, 1, 1, 144)               // two whole partial sums, and one and a half
DENSE_SPLIT_TEST(n, 64, 192, 80, 2, 2, 1, 1, 80)
BGEMM_SPLIT_TEST(o, 2, 64, 192, 64, 1, 4, 4, 1, 64)              // one block of columns a wave, partial sums of two stages and of four
DENSE_SPLIT_TEST(p, 32, 288, 64, 1, 2, 2, 1, 32)
BGEMM_SPLIT_TEST(q, 3, 48, 24, 32, 1, 3, 1, 1, 32)               // one stage, and that not whole
CONV1_SPLIT_TEST(g, 48, 80, 9, 9, 1, 5, 1, 4, 2, 1, 128)
CONV1_SPLIT_TEST(h, 56, 64, 9, 7, 2, 11, 2, 2, 1, 2, 96)
CONV1_SPLIT_TEST(r, 64, 160, 9, 9, 1, 5, 1, 10, 1, 1, 128)       // ten waves, block-fused in the form of five
BFUSE_BFUSE_KERNEL(selftest_gemm_split_r, Narrow<GemmSp_r>, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_gemm_split_a, GemmSp_a, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_HFUSE_KERNEL(selftest_gemm_split_e, GemmSp_e, bias_relu_4096, BiasReluS)
BFUSE_HFUSE_KERNEL(selftest_gemm_split_f, GemmSp_f, conv3x3_f32_32x12x12_32, ConvS2)

// The same products with the first operand taken apart before: _p of a, b, h, i, j, l and r, and a dense one with a last stage of eight k.
#define PARTS_TEST(TAG, OP, I, F, O)                                                                               \
    using GemmSpP_##TAG = OP;                                                                                       \
    BFUSE_KERNEL(selftest_gemm_split_##TAG##_p, GemmSpP_##TAG, (I), (F), (O))
#define DIMS4(...) {{__VA_ARGS__}, 4}
#define PARTS_OF(...) GemmSplit<__VA_ARGS__, false, true>
DENSE_SPLIT_TEST(s, 160, 104, 144, 2, 4, 1, 1, 64)
PARTS_TEST(s, PARTS_OF(160, 104, 1, 144, 1, 1, 2, 4, 1, 1, 64, kPix, 1, 1, 0), DIMS4(160, 104, 1, 1), DIMS4(104, 144, 1, 1), DIMS4(160, 144, 1, 1))
PARTS_TEST(a, PARTS_OF(160, 96, 1, 144, 1, 1, 2, 4, 1, 1, 64, kPix, 1, 1, 0), DIMS4(160, 96, 1, 1), DIMS4(96, 144, 1, 1), DIMS4(160, 144, 1, 1))
PARTS_TEST(b, PARTS_OF(128, 256, 1, 96, 1, 1, 2, 4, 1, 2, 96, kPix, 1, 1, 0), DIMS4(128, 256, 1, 1), DIMS4(256, 96, 1, 1), DIMS4(128, 96, 1, 1))
PARTS_TEST(h, SwapOperands<PARTS_OF(64, 56, 9, 7, 2, 11, 2, 2, 1, 2, 96, kPix, 1, 1, 0)>, DIMS4(11, 56, 9, 7), DIMS4(64, 56, 1, 1), DIMS4(11, 64, 5, 4))
PARTS_TEST(i, SwapOperands<PARTS_OF(64, 144, 9, 7, 1, 5, 2, 2, 1, 1, 64, kPix, 3, 3, 1)>, DIMS4(5, 16, 9, 7), DIMS4(64, 16, 3, 3), DIMS4(5, 64, 9, 7))
PARTS_TEST(j, SwapOperands<PARTS_OF(48, 216, 17, 17, 2, 3, 1, 3, 1, 1, 128, kPix, 3, 3, 0)>, DIMS4(3, 24, 17, 17), DIMS4(48, 24, 3, 3), DIMS4(3, 48, 8, 8))
PARTS_TEST(l, SwapOperands<PARTS_OF(80, 480, 12, 10, 3, 7, 1, 4, 1, 1, 112, kPix, 5, 6, 2)>, DIMS4(7, 16, 12, 10), DIMS4(80, 16, 5, 6), DIMS4(7, 80, 4, 3))
PARTS_TEST(r, SwapOperands<PARTS_OF(160, 64, 9, 9, 1, 5, 1, 10, 1, 1, 128, kPix, 1, 1, 0)>, DIMS4(5, 64, 9, 9), DIMS4(160, 64, 1, 1), DIMS4(5, 160, 9, 9))
BFUSE_BFUSE_KERNEL(selftest_gemm_split_r_p, Narrow<GemmSpP_r>, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)

// Results a line at a time, past the caches, which large ones are (_w): two and six blocks of columns, 16-row blocks, waves over the columns, groups over K, images whose last
// tile is cut, operands taken apart before.
#define LINES_TEST(TAG, I, F, O, WRAP, ...)                                                                         \
    using GemmSpL_##TAG = WRAP<GemmSplit<__VA_ARGS__, 0>>;                                                          \
    using GemmSpW_##TAG = WRAP<GemmSplit<__VA_ARGS__, 1>>;                                                          \
    BFUSE_KERNEL(selftest_gemm_lines_##TAG, GemmSpL_##TAG, (I), (F), (O))                                           \
    BFUSE_KERNEL(selftest_gemm_lines_##TAG##_w, GemmSpW_##TAG, (I), (F), (O))
template <class Op>
using AsItIs = Op;
LINES_TEST(a, DIMS4(3, 128, 72, 1), DIMS4(3, 192, 72, 1), DIMS4(3, 128, 192, 1), AsItIs, 128, 72, 1, 192, 1, 3, 2, 2, 1, 1, 96, kRows, 1, 1, 0, true, false)
LINES_TEST(b, DIMS4(2, 64, 128, 1), DIMS4(2, 128, 128, 1), DIMS4(2, 64, 128, 1), AsItIs, 64, 128, 1, 128, 1, 2, 1, 2, 2, 2, 128, kRows, 1, 1, 0, false, false)
LINES_TEST(c, DIMS4(5, 48, 8, 12), DIMS4(64, 48, 1, 1), DIMS4(5, 64, 8, 12), SwapOperands, 64, 48, 8, 12, 1, 5, 2, 2, 1, 1, 128, kPix, 1, 1, 0, false, false)
LINES_TEST(d, DIMS4(3, 32, 8, 8), DIMS4(160, 32, 3, 3), DIMS4(3, 160, 8, 8), SwapOperands, 160, 288, 8, 8, 1, 3, 1, 10, 1, 1, 128, kPix, 3, 3, 1, false, true)
BFUSE_BFUSE_KERNEL(selftest_gemm_lines_a_w, GemmSpW_a, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_gemm_lines_d_w, Narrow<GemmSpW_d>, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)

// The convolution from a patch taken apart once: pixels that run on into the next images and past the batch, rectangles past an image's
// edges with whole and with broken quads of pixels, one to four groups of channels, units that a thread does twice, two waves over the columns.
// <CI, CO, H, W, padding, images, 16-row blocks of a wave, waves over rows, over columns, pixels, width>
#define CONV_PATCH_TEST(TAG, CI, CO, H, W, P, N, ...)                                                              \
    using ConvP_##TAG = SwapOperands<ConvSplit<CI, CO, H, W, 3, 3, 1, P, N, __VA_ARGS__>>;                          \
    BFUSE_KERNEL(selftest_conv_split_##TAG, ConvP_##TAG, ({{N, CI, H, W}, 4}), ({{CO, CI, 3, 3}, 4}), ({{N, CO, H - 2 + 2 * P, W - 2 + 2 * P}, 4}))
CONV_PATCH_TEST(a, 64, 64, 7, 7, 1, 5, 2, 2, 1, 96, 0)           // 245 pixels of five images in three tiles
CONV_PATCH_TEST(b, 32, 96, 13, 15, 1, 2, 2, 3, 1, 144, 12)       // one group, rectangles of 12 x 12 on 13 x 15
CONV_PATCH_TEST(c, 96, 256, 30, 18, 0, 2, 2, 4, 1, 112, 28)      // rectangles of 28 on 16 columns, two row tiles
CONV_PATCH_TEST(d, 32, 32, 20, 33, 1, 2, 2, 1, 2, 224, 16)
CONV_PATCH_TEST(e, 128, 128, 10, 10, 0, 4, 2, 4, 2, 224, 0)      // 256 pixels of four images
CONV_PATCH_TEST(f, 64, 64, 9, 9, 2, 3, 2, 2, 1, 112, 16)         // padding of two
CONV_PATCH_TEST(g, 96, 128, 5, 5, 1, 9, 2, 4, 1, 128, 0)         // a tile of six images
CONV_PATCH_TEST(h, 160, 64, 7, 7, 1, 5, 2, 2, 1, 96, 0)          // five groups of channels: partial sums of three taps
BFUSE_BFUSE_KERNEL(selftest_conv_split_a, ConvP_a, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_HFUSE_KERNEL(selftest_conv_split_b, ConvP_b, bias_relu_4096, BiasReluS)
BFUSE_HFUSE_KERNEL(selftest_conv_split_d, ConvP_d, conv3x3_f32_32x12x12_32, ConvS2)
BFUSE_BFUSE_RT_KERNEL(selftest_conv_split_f, ConvP_f, layernorm_8x256, LayerNormS)
// (beside ten waves: 168 registers)
BFUSE_BFUSE_KERNEL(selftest_conv_split_a, Slim<ConvP_a>, gemm_bf16_256x448x1792_p2, GemmB9, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_conv_split_b, Slim<ConvP_b>, gemm_bf16_256x448x1792_p2, GemmB9, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_conv_split_d, Slim<ConvP_d>, gemm_bf16_256x448x1792_p2, GemmB9, _c4, bfuse::kChunked, 4, 1)
BFUSE_BFUSE_KERNEL(selftest_conv_split_a, ConvP_a, selftest_gemm_split_r_p, Narrow<GemmSpP_r>, _c4, bfuse::kChunked, 4, 1)   // operands of both sides are taken apart

// The split-K product on the bf16 matrix cores: a trailing 16-column group and GELU in one round, two waves in two rounds, one stage; 32
// and 48 columns past the last group.
using GemmSpk_a = GemmF32Dma<64, 288, 256, 32, 144, 4, kEpiGeluTanh>;
using GemmSpk_b = GemmF32Dma<96, 256, 192, 32, 128, 2, kEpiNone, 2>;
using GemmSpk_c = GemmF32Dma<32, 384, 128, 32, 192, 4, kEpiNone, 2>;
using GemmSpk_d = GemmSplitK<64, 288, 192, 32, 96, 2, kEpiNone, 1>;
using GemmSpk_e = GemmSplitK<64, 336, 256, 32, 112, 4, kEpiNone, 2>;
BFUSE_KERNEL(selftest_gemm_splitk_a, GemmSpk_a, ({{64, 256, 1, 1}, 4}), ({{256, 288, 1, 1}, 4}), ({{64, 288, 1, 1}, 4}))
BFUSE_KERNEL(selftest_gemm_splitk_b, GemmSpk_b, ({{96, 192, 1, 1}, 4}), ({{192, 256, 1, 1}, 4}), ({{96, 256, 1, 1}, 4}))
BFUSE_KERNEL(selftest_gemm_splitk_c, GemmSpk_c, ({{32, 128, 1, 1}, 4}), ({{128, 384, 1, 1}, 4}), ({{32, 384, 1, 1}, 4}))
BFUSE_KERNEL(selftest_gemm_splitk_d, GemmSpk_d, ({{64, 192, 1, 1}, 4}), ({{192, 288, 1, 1}, 4}), ({{64, 288, 1, 1}, 4}))
BFUSE_KERNEL(selftest_gemm_splitk_e, GemmSpk_e, ({{64, 256, 1, 1}, 4}), ({{256, 336, 1, 1}, 4}), ({{64, 336, 1, 1}, 4}))
BFUSE_BFUSE_KERNEL(selftest_gemm_splitk_a, GemmSpk_a, layernorm_8x256, LayerNormS, _c4, bfuse::kChunked, 4, 1)
BFUSE_HFUSE_KERNEL(selftest_gemm_splitk_b, GemmSpk_b, bias_relu_4096, BiasReluS)
BFUSE_HFUSE_KERNEL(selftest_gemm_splitk_b, GemmSpk_b, conv3x3_f32_32x12x12_32, ConvS2)
