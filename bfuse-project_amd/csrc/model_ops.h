// The operators of the reference's example models as the library instantiates them: one alias per operator id
// (test-utils/examples/llm.yaml, resnet-18.yaml).  A fused kernel and the standalone kernel it is compared
// with must be built from the SAME instantiation, so every file that names one of these takes it from here.
#pragma once
#include "ops_conv.h"
#include "ops_conv_few.h"
#include "ops_conv_general.h"
#include "ops_conv_rect.h"
#include "ops_gemm_bf16.h"
#include "ops_gemm_f32.h"
#include "ops_gemm_f32_dma.h"
#include "ops_gemm_split.h"
#include "ops_gemm_tile.h"
#include "ops_rowwise.h"

namespace bfuse {
namespace model {

// dense_0: BERT attention output projection, [512 x 768] . [768 x 768]: 16 x 16 tiles of 32 x 48
using Dense0 = GemmF32Dma<512, 768, 768, 32, 48, 4>;
// dense_1: BERT / GPT-2 MLP up-projection without the activation, [512 x 768] . [768 x 3072]: pair 4's tiling
using Dense1 = GemmF32Dma<512, 3072, 768, 32, 96, 4, kEpiNone, 2>;
// dense_2: MLP down-projection, [512 x 3072] . [3072 x 768]: two stages of 16 k in the ring (40 KB: four workgroups of a fused
// kernel per CU; three stages are 0.1 us faster alone and 3 us slower fused with attention products)
using Dense2 = GemmF32Dma<512, 768, 3072, 32, 48, 4, kEpiNone, 2>;
// dense_3: the QKV projection of pair 2
using Dense3 = GemmF32Dma<512, 2304, 768, 32, 144, 4>;
// dense_4 / dense_7 (Llama-3-8B, bf16, weights [N, K]): N = 4096 over 256 CUs leaves each a 64 x 128 tile: four
// compute waves (2 x 2) of 32 x 64 and two producer waves, ring of four 64-k stages (96 KB), read-ahead of two
// fragments, the next step's barrier before MFMA group 6 of 8.  A stage is 24 KB for 256 clocks of MFMAs: what bounds the
// layer is how many bytes are under way, 72 KB with four stages.  Three: 71.9 against 67.0 us (K = 14336) and 23.8 against
// 22.5, and although two workgroups of three stages fit a CU the fusions gain as well (with the norm 76.6 -> 71.6 and
// 28.6 -> 26.3, with convolutions 1.04-1.05x).  Five and six stages are like four (66.8, 67.5; 22.5, 22.0), 128 x 128 tiles
// on half the CUs 77.8 and 24.3.
using Dense4 = GemmBf16NTDma<512, 4096, 4096, 64, 128, 4, 2, 2, 2, 2, 6>;
using Dense7 = GemmBf16NTDma<512, 4096, 14336, 64, 128, 4, 2, 2, 2, 2, 6>;
// dense_5: Llama-3-8B key / value projection, [512 x 4096] . [4096 x 1024]: 16 x 16 tiles of 32 x 64
using Dense5 = GemmF32Dma<512, 1024, 4096, 32, 64, 4>;
// dense_6: the gate projection of pair 5
using Dense6 = GemmBf16NTDma<512, 14336, 4096, 128, 224, 3, 4, 4, 2, 2, 11>;

// Batched GEMMs of the attention layers (the reference's bgemm, scripts/configure_kernels.py:14-19,40-48:
// C[b] = A[b] . B[b]^T with A [b, M, K] and B [b, N, K]): bgemm_0 / bgemm_1 are BERT's and GPT-2's scores and
// context products (12 heads, sequence 512, head size 64), bgemm_2 / bgemm_3 Llama-3-8B's (32 heads, head size 128).
// bgemm_1 has 8 row tiles a product, too few of 64 rows (12.2 us): operands go global -> VGPR in MFMA layout, two waves split K.
// (32 x 64 two-wave 9.7 us, 16 x 64 two-wave 11.3, four-wave 11.3, 16 x 32 10.1.)  Split into bf16 (GemmSplit, 64 x 32 tiles) it takes
// 8.0, but beside the bf16 product's hand-counted reads the compiler then moves registers in a way that the build's check refuses.
// The others run on the bf16 matrix cores (GemmSplit).  us alone and fused with the fp32 768 x 768, 768 x 3072 and 768 x 2304 and the bf16
// 4096 x 4096 and 4096 x 14336 layers, fp32 matrix cores (GemmTile) before:
//   bgemm_0  6.8, 12.4, 25.3, 21.1, 27.4, 52.6 -> 6.2, 11.8, 23.7, 19.8, 27.6, 52.8, with the causal softmax 9.6 -> 8.5; 64 x 64 tiles of four
//            16-row waves (lean 6.05, 11.6, 23.3, 19.4, but 27.6 and 53.3; 128 x 64 of 32-row waves 7.4)
//   bgemm_2  21.4, 29.2, 42.4, 36.9, 46.1, 73.2 -> 17.4, 22.2, 39.6, 32.6, 37.7, 63.6; 128 x 128 tiles of eight 16-row waves (128 x 64 of four
//            32-row waves 18.2, 24.1, 36.3, 29.7, 40.2, 65.1)
//   bgemm_3  20.1 alone, 33.0, 42.5, 67.3 with the last three -> 16.4, 27.8, 34.9, 61.1; 128 x 64 tiles of four 32-row waves (lean 17.9, 28.1, 36.6, 62.4, and with the
//            768 x 768 and 3072 x 768 layers 22.7, 34.9 -> 21.4, 33.9).  The twelve waves a CU of a fused kernel with the bf16 gate projection leave 168 registers: 163
using Bgemm0 = GemmSplit<512, 64, 1, 512, 1, 12, 1, 4, 1, 1, 64, kRows, 1, 1, 0, false>;      // 8 x 8 tiles x 12 = 768 workgroups
using Bgemm1 = GemmF32<512, 64, 512, 32, 64, 2, kEpiNone, 2, 1, true, 12>;     // 16 x 1 tiles x 12 = 192 two-wave workgroups
using Bgemm2 = GemmSplit<512, 128, 1, 512, 1, 32, 1, 8, 1, 1, 128, kRows>;                    // 4 x 4 tiles x 32 = 512
using Bgemm3 = GemmSplit<512, 512, 1, 128, 1, 32, 2, 4, 1, 1, 64, kRows, 1, 1, 0, false>;     // 4 x 2 tiles x 32 = 256

// conv2d_1: the convolution of pair 3;  conv2d_4: 128 -> 128 channels on 28 x 28, 32 output channels x 16 pixels
// per workgroup, four waves take two 16-channel groups each, 49 x 4 = 196 workgroups (eight waves on 16 channels x 32 pixels:
// 6.9 us alone against 8.9, but fused with the dense layers of two workgroups per CU 28.7 against 26.3)
using Conv1 = Conv3x3F32Lds<64, 64, 56, 56, 16, 4, 4>;
using Conv4 = Conv3x3F32Lds<128, 128, 28, 28, 32, 1, 4>;

// fp32 instantiations of the Llama-3-8B layers (the reference computes every layer in fp32), on the bf16 matrix cores: 256
// tiles of 128 x 64 for N = 4096 (dense_4, dense_7: 119 -> 93 us, 404 -> 308) and of 256 x 112 for N = 14336 (dense_6: 461 ->
// 254; two groups of waves over K on 128 x 112 tiles 282), with the activations taken apart before 95 -> 91, 324 -> 309, 263 -> 259.  Before: GemmF32Dma on 64 x 128 tiles.
using Dense4F32 = GemmSplit<512, 4096, 1, 4096, 1, 1, 2, 4, 1, 2, 64, kPix, 1, 1, 0, false, true>;
using Dense6F32 = GemmSplit<512, 4096, 1, 14336, 1, 1, 2, 8, 1, 1, 112, kPix, 1, 1, 0, false, true>;
using Dense7F32 = GemmSplit<512, 14336, 1, 4096, 1, 1, 2, 4, 1, 2, 64, kPix, 1, 1, 0, false, true>;

// bgemm_4 .. bgemm_17 of llm.yaml (ViT / Swin / small-model attention products: 16 heads x 256 or 208 tokens with
// head sizes 64 and 80, and single-head products of 512 / 768 / 1024 tokens).  Scores (reductions of 64 and 80) run on
// shared 64 x 64 tiles, four waves for each of 128 - 256 tiles where one wave had it before: 6.1 -> 3.8 us, 7.0 -> 4.4, with
// 208 rows and columns (the last tiles overlap) 5.5 -> 3.6, 6.2 -> 4.3, one head of 1024 3.9 -> 3.3; the same bits.  Context
// products have one column tile a product and too few row tiles for that (256 x 256 x 64: 6.8 against 4.3 us): 208 = 13 x 16
// and 80 = 5 x 16 are whole 16-wide MFMA blocks, an 80-column tile is one 64-column group and one of 16; a reduction of 208 is
// thirteen 16-k stages of one wave.
using Bgemm4 = GemmTile<256, 64, 1, 256, 1, 16, 64, 64, 4, 32, kRows, 2>;      // 4 x 4 tiles x 16 = 256 workgroups
using Bgemm5 = GemmF32<256, 64, 256, 16, 64, 2, kEpiNone, 2, 1, true, 16>;      // 16 x 1 x 16 = 256 two-wave workgroups
using Bgemm6 = GemmTile<256, 80, 1, 256, 1, 16, 64, 64, 4, 16, kRows, 2>;
using Bgemm7 = GemmF32<256, 80, 256, 16, 80, 2, kEpiNone, 2, 1, true, 16>;
using Bgemm8 = GemmTile<208, 64, 1, 208, 1, 16, 64, 64, 4, 32, kRows, 2>;      // 4 x 4 overlapping tiles x 16
using Bgemm9 = GemmF32<208, 64, 208, 16, 64, 1, kEpiNone, 2, 1, true, 16>;
using Bgemm10 = GemmTile<208, 80, 1, 208, 1, 16, 64, 64, 4, 16, kRows, 2>;
using Bgemm11 = GemmF32<208, 80, 208, 16, 80, 1, kEpiNone, 2, 1, true, 16>;
using Bgemm12 = GemmF32<512, 256, 64, 16, 64, 1, kEpiNone, 2, 1, true, 1>;      // 32 x 4 = 128 one-wave workgroups
using Bgemm13 = GemmF32<512, 64, 256, 16, 64, 4, kEpiNone, 2, 1, true, 1>;      // 32 four-wave workgroups
using Bgemm14 = GemmF32<768, 384, 64, 16, 64, 1, kEpiNone, 2, 1, true, 1>;      // 48 x 6 = 288
using Bgemm15 = GemmF32<768, 64, 384, 16, 64, 4, kEpiNone, 2, 1, true, 1>;      // 48 four-wave workgroups
using Bgemm16 = GemmTile<1024, 64, 1, 512, 1, 1, 64, 64, 4, 32, kRows, 2>;      // 16 x 8 = 128
using Bgemm17 = GemmF32<1024, 64, 512, 16, 64, 4, kEpiNone, 2, 1, true, 1>;     // 64 four-wave workgroups

// The other ResNet-18 layers (test-utils/examples/resnet-18.yaml) on the general convolution:
// <CI, CO, H, W, KH, KW, stride, padding, output channels per workgroup, 16-pixel blocks, waves>
// One image has 128 - 208 tiles of 16 x 16 results and a reduction of 576 - 4608 for each: staging and the chain of MFMAs
// of a wave are what takes the time, so the 3x3 layers of 128 channels and more split it over eight waves.  us with eight: 512 channels on 7x7 8.6, 256 on
// 14x14 5.5, 256 -> 512 and 128 -> 256 at stride 2 6.1 and 4.3.  (Against four waves, measured while filters came as the lanes want them and these took
// 14.7, 8.9, 9.9 and 6.5: 1.16x, 1.12x, 1.15x and 1.05x, sixteen waves on 7x7 1.01x more, but 0.91x fused with the LayerNorm; the 1x1 layers gained 1.1-1.2x
// alone and lost 0.74-0.84x fused: four waves.)
using Conv0 = ConvF32Few<3, 64, 224, 224, 7, 7, 2, 3, 16, 4, 1>;          // 7x7 stride 2 on RGB: 4 x 16-pixel rectangles (13 x 37 patch instead of 9 x 230), 196 x 4 = 784 one-wave workgroups
using Conv2 = SwapOperands<GemmF32<64, 3136, 64, 16, 64, 1>>;            // 1x1 stride 1 = Wt[64,64] . X[64,3136]: 4 x 49 = 196
using Conv3 = ConvF32Lds<64, 128, 56, 56, 3, 3, 2, 1, 16, 2, 4>;          // 25 x 8 = 200 workgroups; 32 channels x 16 pixels 1.05x the time, fused 1.35x
using Conv5 = ConvF32Lds<64, 128, 56, 56, 1, 1, 2, 0, 32, 1, 4>;
using Conv6 = ConvF32Lds<128, 256, 28, 28, 3, 3, 2, 1, 16, 1, 8>;         // 13 x 16 = 208
using Conv7 = ConvF32Lds<256, 256, 14, 14, 3, 3, 1, 1, 16, 1, 8>;
using Conv8 = ConvF32Lds<128, 256, 28, 28, 1, 1, 2, 0, 16, 1, 4>;
using Conv9 = ConvF32Lds<256, 512, 14, 14, 3, 3, 2, 1, 16, 1, 8>;         // 4 x 32 = 128
using Conv10 = ConvF32Lds<512, 512, 7, 7, 3, 3, 1, 1, 16, 1, 8>;
using Conv11 = ConvF32Lds<256, 512, 14, 14, 1, 1, 2, 0, 16, 1, 4>;

// memory-bound partners
using LayerNormW1 = LayerNorm<512, 768, 1, 1>;
using NormRopeW1 = RmsNormRope<512, 32, 128, 1>;
using Softmax4W = SoftmaxCausal<12, 512, 4, 1>;

}  // namespace model
}  // namespace bfuse
