"""The shared-tile convolution and product (csrc/ops_conv_tile.h, ops_gemm_tile.h), the dense product's long stages
(ops_gemm_f32_dma.h) and the bf16 product's ring of four (ops_gemm_bf16.h) at the edges of their tiles, against the CPU
oracle (products: numpy in double), alone and fused."""
import numpy as np
import pytest
import torch

import bfuse_project_amd as bf
from bfuse_project_amd.operation import bf16_to_f32, f32_to_bf16, fill_normal
from oracle import oracle as orf
from tests import oracle_cases

pytestmark = pytest.mark.gpu


def _check(name, reference, partner, kind, suffix):
    with bf.Operation(name, partner) as op:
        k, q = op.k
        x, w = fill_normal(3, int(np.prod(k.shapes[0])), 0, 1), fill_normal(4, int(np.prod(k.shapes[1])), 0, 0.1)
        x2, w2 = fill_normal(5, int(np.prod(q.shapes[0])), 0, 1), fill_normal(6, int(np.prod(q.shapes[1])), 0, 1)
        op.upload(0, x, w)
        op.upload(1, x2, w2)
        op.zero_outputs()
        op.launch("serial")
        y, y2 = op.download(0), op.download(1)
        want = reference(x.reshape(k.shapes[0]), w.reshape(k.shapes[1]))
        assert y.size == want.size
        assert oracle_cases.rel_error(y.ravel(), want.ravel()) <= 1e-5
        if kind:
            op.zero_outputs()
            op.launch(kind, op.fused(kind, suffix))
            assert np.array_equal(op.download(0).view(np.uint32), y.view(np.uint32)) and np.array_equal(op.download(1).view(np.uint32), y2.view(np.uint32))


@pytest.mark.parametrize("tag,s,p,partner,kind,suffix", [
    ("a", 1, 1, "bias_relu_4096", "hfuse", ""), ("b", 2, 0, "layernorm_8x256", "bfuse", "_c4"),
    ("c", 1, 2, "conv3x3_f32_32x12x12_32", "hfuse", ""), ("d", 4, 1, "bias_relu_4096", None, ""), ("e", 1, 1, "bias_relu_4096", None, ""),
    ("f", 1, 1, "bias_relu_4096", None, ""), ("g", 1, 1, "bias_relu_4096", None, ""), ("h", 1, 1, "bias_relu_4096", None, "")])
def test_shared_tile_convolution_against_the_oracle_and_fused(tag, s, p, partner, kind, suffix):
    _check(f"selftest_conv_tile_{tag}", lambda x, w: orf.conv2d(x, w, s=s, p=p), partner, kind, suffix)


@pytest.mark.parametrize("tag,s,partner,kind,suffix", [
    ("a", 1, "bias_relu_4096", None, ""), ("b", 1, "bias_relu_4096", None, ""), ("c", 2, "bias_relu_4096", "hfuse", ""), ("d", 1, "bias_relu_4096", None, "")])
def test_shared_tile_1x1_convolution_against_the_oracle_and_fused(tag, s, partner, kind, suffix):
    _check(f"selftest_gemm_tile_{tag}", lambda x, w: orf.conv2d(x, w, s=s, p=0), partner, kind, suffix)


@pytest.mark.parametrize("tag,partner,kind,suffix", [("e", "layernorm_8x256", "bfuse", "_c4"), ("f", "bias_relu_4096", None, ""), ("g", "bias_relu_4096", None, "")])
def test_shared_tile_batched_product_against_numpy_and_fused(tag, partner, kind, suffix):
    def product(a, b):
        return np.matmul(a[..., 0].astype(np.float64), b[..., 0].astype(np.float64).transpose(0, 2, 1)).astype(np.float32)
    _check(f"selftest_gemm_tile_{tag}", product, partner, kind, suffix)


@pytest.mark.parametrize("name,steps,parts", [("selftest_conv_tile_h", 64 * 9 // 4, 16 / 3), ("selftest_gemm_tile_g", 512 // 4, 2)])
def test_long_reductions_are_summed_in_parts(name, steps, parts):
    """A sum of random terms that is rounded after each of `steps` steps, by at most u = 2^-24 of what it has grown to, is
    off by at most u sqrt(steps / 2) of the result (2-norm); in `parts` equal parts by sqrt(parts) less.  (In one sum these
    two are 3.0e-7 and 4.1e-7 off, the bounds are 2.2e-7 and 3.4e-7.)"""
    with bf.Operation(name, "bias_relu_4096") as op:
        k = op.k[0]
        x, w = (fill_normal(7 + i, int(np.prod(k.shapes[i])), 0, 1).reshape(k.shapes[i]) for i in (0, 1))
        op.upload(0, x, w)
        op.launch("kernel1")
        y = op.download(0).ravel().astype(np.float64)
    if "conv" in name:
        want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), padding=1).numpy()
    else:
        want = np.matmul(x[..., 0].astype(np.float64), w[..., 0].astype(np.float64).transpose(0, 2, 1))
    assert np.linalg.norm(y - want.ravel()) <= 2.0 ** -24 * (steps / 2 / parts) ** 0.5 * np.linalg.norm(want)


def test_long_stages_of_the_dense_product_against_numpy_and_fused():
    _check("selftest_gemm_long", lambda a, b: (a[..., 0, 0].astype(np.float64) @ b[..., 0, 0].astype(np.float64)).astype(np.float32),
           "bias_relu_4096", "hfuse", "")


def test_ring_of_four_stages_of_the_bf16_product_against_numpy():
    """Operands are bf16, sums fp32: what is left is the rounding of the result to eight bits (half a unit in the last place
    is at most 2^-8 of it) and 1e-5 of the sum's size."""
    with bf.Operation("selftest_gemm_ring4", "bias_relu_4096") as op:
        k = op.k[0]
        a, b = (f32_to_bf16(fill_normal(8 + i, int(np.prod(k.shapes[i])), 0, 1)) for i in (0, 1))
        op.upload(0, a, b)
        op.launch("kernel1")
        y = bf16_to_f32(op.download(0)).reshape(128, 1024).astype(np.float64)
    want = bf16_to_f32(a).reshape(128, 704).astype(np.float64) @ bf16_to_f32(b).reshape(1024, 704).astype(np.float64).T
    assert np.all(np.abs(y - want) <= 2.0 ** -8 * np.abs(want) * (1 + 1e-5) + 1e-5 * np.sqrt(704))
