// The dense and bgemm operators of the reference's test-utils/examples/benchmark.yaml: the layers of llm.yaml at
// 1024 rows (dense: batch, in, out) and at 1024 independent products (bgemm: batch, M, K, N), fp32, with the
// tilings of their 512-row / 16-product counterparts (model_ops.h) -- twice, or 64 times, the workgroups -- or with twice
// the columns per tile, which is again a workgroup per CU and a better ratio of MFMAs to operand reads: 1024 x 3072 x 768
// 44.4 -> 34.8 us (32 x 96 against 32 x 48), x 768 x 768 11.5 -> 10.8, 4096 x 1024 62.5 -> 60.2 (32 x 128 against 32 x 64).  The larger ones run on the bf16 matrix cores (ops_gemm_split.h has the figures): there the
// tile is 128 x 128, 128 x 96 or 256 x 112 (two whole rounds for 14336 columns; 128 are one and three quarters), the largest that still gives every CU one.  Those that have no 256 such tiles split K over the
// waves of 32 x 96 - 32 x 144 tiles instead (GemmF32Dma): 1024 x 768 x 2304 24.8 us, on 192 tiles of 128 x 96 30.2.
#include "fuse.h"
#include "ops_gemm_f32.h"
#include "ops_gemm_f32_dma.h"
#include "ops_gemm_split.h"

using namespace bfuse;

BFUSE_MODULE_PROLOGUE()

#define DENSE_F32(M, K, N, ...)                                                                                  \
    using Dense_##M##x##K##x##N = GemmF32Dma<M, N, K, __VA_ARGS__>;                                               \
    BFUSE_KERNEL(gemm_f32_##M##x##K##x##N, Dense_##M##x##K##x##N, ({{M, K, 1, 1}, 4}), ({{K, N, 1, 1}, 4}), ({{M, N, 1, 1}, 4}))
// <.., 16-row blocks of a wave, waves over the rows, over the columns, over K, columns>
#define DENSE_SPLIT(M, K, N, ...)                                                                                \
    using Dense_##M##x##K##x##N = GemmSplit<M, K, 1, N, 1, 1, __VA_ARGS__>;                                       \
    BFUSE_KERNEL(gemm_f32_##M##x##K##x##N, Dense_##M##x##K##x##N, ({{M, K, 1, 1}, 4}), ({{K, N, 1, 1}, 4}), ({{M, N, 1, 1}, 4}))
DENSE_F32(1024, 768, 768, 32, 96, 4)
DENSE_SPLIT(1024, 768, 3072, 2, 4, 1, 2, 96, kPix)
DENSE_F32(1024, 3072, 768, 32, 96, 4)
DENSE_F32(1024, 768, 2304, 32, 144, 4)
DENSE_SPLIT(1024, 4096, 4096, 2, 4, 1, 2, 128, kPix)
DENSE_F32(1024, 4096, 1024, 32, 128, 4)
DENSE_SPLIT(1024, 4096, 14336, 2, 8, 1, 1, 112, kPix, 1, 1, 0, false, true)
DENSE_SPLIT(1024, 14336, 4096, 2, 4, 1, 2, 128, kPix)

// C[b] = A[b] . B[b]^T, A [b, M, K], B [b, N, K].  Those of 208 rows: <M, N, K, BM, BN, waves over K>, a tile per wave; the one-wave
// products reserve 32 KB of LDS per workgroup: four workgroups per CU, one wave per SIMD (see LdsReserve).
#define BGEMM_F32_RESERVE(B, M, K, N, BM, BN, KS, BYTES)                                                         \
    using Bgemm_##B##x##M##x##K##x##N = LdsReserve<GemmF32<M, N, K, BM, BN, KS, kEpiNone, 2, 1, true, B>, BYTES>; \
    BFUSE_KERNEL(bgemm_f32_##B##x##M##x##K##x##N, Bgemm_##B##x##M##x##K##x##N, ({{B, M, K, 1}, 4}), ({{B, N, K, 1}, 4}), ({{B, M, N, 1}, 4}))
// The bf16 matrix cores (ops_gemm_split.h): 128 x 64 tiles of 32-row waves for the long reductions, 128 x 128 of eight 16-row waves for
// those of 64 - 128, which are mostly ends: 70 - 94 registers instead of 126 - 168, so that three workgroups a CU load, multiply and
// store at different times.  us on one card, fp32 matrix cores before and now: 1024 products 512 x 64 x 512 360 -> 303 (32-row waves 311-348), 512 x
// 128 x 512 625 -> 465 (499), 256 x 64 x 256 98 -> 84 (94), 256 x 80 x 256 119 -> 107 (117), 1024 x 64 x 512 705 -> 609 (620), 256 x 256 x
// 80 134 -> 95 (16-row waves; 32-row 99), 512 x 512 x 128 555 -> 416 (32-row, 128 x 128, lean; not lean 424, 16-row 446), 512 x 512 x 64 334 -> 268 (293), 1024 x
// 512 x 64 607 -> 518 (573), 256 x 256 x 64 95.6 -> 83 (88).  Results of more than 256 MB
// since go past the caches in whole lines (GemmSplit, LINES): 512 x 64 x 512 308 -> 270, 512 x 128 x 512 468 -> 458, 1024 x 64 x 512 602 -> 579.  208 x 208 x 64 gains nothing (75.9 against 74); 208 x 64 x 208, x 80 x 208
// and x 208 x 80 gain 1.1-1.4x on seven or thirteen waves but keep the one-wave forms, which any operator can take beside it.
#define BGEMM_F32_SPLIT(B, M, K, N, ...)                                                                         \
    using Bgemm_##B##x##M##x##K##x##N = GemmSplit<M, K, 1, N, 1, B, __VA_ARGS__>;                                 \
    BFUSE_KERNEL(bgemm_f32_##B##x##M##x##K##x##N, Bgemm_##B##x##M##x##K##x##N, ({{B, M, K, 1}, 4}), ({{B, N, K, 1}, 4}), ({{B, M, N, 1}, 4}))
BGEMM_F32_SPLIT(1024, 512, 64, 512, 1, 8, 1, 1, 128, kRows)
BGEMM_F32_SPLIT(1024, 512, 512, 64, 2, 4, 1, 1, 64, kRows)
BGEMM_F32_SPLIT(1024, 512, 128, 512, 1, 8, 1, 1, 128, kRows)
BGEMM_F32_SPLIT(1024, 512, 512, 128, 2, 4, 1, 1, 128, kRows, 1, 1, 0, true)
BGEMM_F32_SPLIT(1024, 256, 64, 256, 1, 8, 1, 1, 128, kRows)
BGEMM_F32_SPLIT(1024, 256, 256, 64, 2, 4, 1, 1, 64, kRows)
BGEMM_F32_SPLIT(1024, 256, 80, 256, 1, 8, 1, 1, 128, kRows)
BGEMM_F32_SPLIT(1024, 256, 256, 80, 1, 8, 1, 1, 80, kRows)
BGEMM_F32_RESERVE(1024, 208, 64, 208, 112, 64, 1, 32768)
BGEMM_F32_RESERVE(1024, 208, 208, 64, 208, 32, 1, 32768)
BGEMM_F32_RESERVE(1024, 208, 80, 208, 112, 64, 1, 32768)     // 208 = 112 + 96 rows, 3 x 64 + 16 columns: the last tiles overlap their neighbours
BGEMM_F32_RESERVE(1024, 208, 208, 80, 64, 80, 1, 32768)
// tests/interleave_scheduler/config/info.yaml: bgemm_6, bgemm_7
BGEMM_F32_SPLIT(1024, 1024, 64, 512, 1, 8, 1, 1, 128, kRows)
BGEMM_F32_SPLIT(1024, 1024, 512, 64, 2, 4, 1, 1, 64, kRows)
