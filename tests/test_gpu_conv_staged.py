"""The convolutions whose waves stage a patch of their own (csrc/ops_conv.h, ops_conv_general.h, ops_conv_rect.h, ops_conv_few.h) and take their filters through
LDS (ops_conv_filters.h), at the edges of images, vectors, row blocks and groups, against the oracle; three of them fused, bit for bit."""
import numpy as np
import pytest
import torch

import bfuse_project_amd as bf
from bfuse_project_amd.operation import f32_to_bf16, fill_normal
from oracle import oracle as orf
from tests.test_gpu_conv_tile import _check

pytestmark = pytest.mark.gpu

FORMS = [("a", 1, 2, "bias_relu_4096", "hfuse", ""), ("b", 1, 1, "bias_relu_4096", None, ""), ("c", 2, 1, "bias_relu_4096", None, ""), ("d", 1, 5, "bias_relu_4096", None, ""),
         ("e", 1, 0, "bias_relu_4096", None, ""), ("f", 2, 3, "bias_relu_4096", None, ""), ("g", 1, 1, "layernorm_8x256", "bfuse", "_c4"), ("h", 2, 1, "bias_relu_4096", None, ""),
         ("i", 1, 2, "bias_relu_4096", None, ""), ("j", 1, 1, "bias_relu_4096", None, ""), ("k", 1, 1, "bias_relu_4096", None, ""), ("l", 1, 1, "bias_relu_4096", "hfuse", ""),
         ("m", 1, 0, "bias_relu_4096", "hfuse", ""), ("n", 2, 2, "bias_relu_4096", None, ""), ("o", 1, 1, "bias_relu_4096", None, ""), ("p", 2, 3, "bias_relu_4096", None, ""),
         ("q", 1, 7, "bias_relu_4096", None, ""), ("r", 1, 6, "bias_relu_4096", None, ""), ("s", 1, 3, "bias_relu_4096", None, ""),
         ("t", 5, 0, "bias_relu_4096", "hfuse", ""), ("u", 5, 2, "conv3x3_f32_32x12x12_32", "hfuse", ""), ("v", 8, 0, "conv3x3_f32_32x12x12_32", "hfuse", ""),
         ("w", 4, 1, "bias_relu_4096", None, ""), ("x", 1, 17, "bias_relu_4096", None, ""), ("y", 1, 35, "bias_relu_4096", None, ""), ("z", 1, 18, "bias_relu_4096", None, ""),
         ("aa", 1, 67, "bias_relu_4096", None, ""), ("ba", 1, 2, "bias_relu_4096", None, ""), ("bb", 1, 2, "bias_relu_4096", None, ""), ("bc", 1, 1, "bias_relu_4096", None, ""),
         ("bd", 2, 1, "bias_relu_4096", None, ""), ("be", 1, 1, "bias_relu_4096", None, ""), ("ca", 4, 6, "bias_relu_4096", None, ""), ("cb", 1, 0, "bias_relu_4096", None, ""),
         ("da", 1, 0, "bias_relu_4096", None, ""), ("db", 1, 4, "bias_relu_4096", None, ""), ("dc", 3, 4, "bias_relu_4096", None, ""), ("dd", 1, 1, "bias_relu_4096", None, "")]


@pytest.mark.parametrize("tag,s,p,partner,kind,suffix", FORMS)
def test_staged_convolution_against_the_oracle_and_fused(tag, s, p, partner, kind, suffix):
    _check(f"selftest_conv_staged_{tag}", lambda x, w: orf.conv2d(x, w, s=s, p=p), partner, kind, suffix)


@pytest.mark.parametrize("tag,s,p", [f[:3] for f in FORMS])
def test_staged_convolution_copies_what_a_selector_names(tag, s, p):
    """Filters of a single one: every result is one (padded) element of the image exactly, at every edge."""
    with bf.Operation(f"selftest_conv_staged_{tag}", "bias_relu_4096") as op:
        k = op.k[0]
        (co, ci, kh, kw), x = k.shapes[1], fill_normal(7, int(np.prod(k.shapes[0])), 0, 1)
        c = np.arange(co)
        w = np.zeros((co, ci, kh, kw), np.float32)
        w[c, (5 * c + 1) % ci, (3 * c) % kh, (2 * c + c // kh) % kw] = 1
        y = op.run_kernel(0, x, w.ravel())
    assert np.array_equal(y.ravel(), orf.conv2d(x.reshape(k.shapes[0]), w, s=s, p=p).ravel())


@pytest.mark.parametrize("tag,s,p", [f[:3] for f in FORMS if f[0] in (*"acdfmnopqrsvwz", "aa", "bb", "ca", "cb")])
def test_a_value_that_is_not_finite_is_in_its_own_windows_alone(tag, s, p):
    """Four k of an MFMA are rows or taps of a window: those that there are not have no part in it, whatever lies in their place."""
    name = f"selftest_conv_staged_{tag}"
    with bf.Operation(name, "bias_relu_4096") as op:
        k = op.k[0]
        x, w = (fill_normal(8 + i, int(np.prod(k.shapes[i])), 0, 1).reshape(k.shapes[i]) for i in (0, 1))
        w = np.abs(w) + np.float32(0.5)
        x[0, 0, 2, 3], x[-1, -1, -1, -1], x[0, -1, 5, 9] = np.inf, np.nan, -np.inf
        y = op.run_kernel(0, x, w).reshape(k.shapes[2])
    with np.errstate(all="ignore"):
        want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), stride=s, padding=p).numpy()
    assert np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(np.isposinf(y), np.isposinf(want)) and np.array_equal(np.isneginf(y), np.isneginf(want))
    ok = np.isfinite(want)
    assert ok.any() and np.linalg.norm(y[ok] - want[ok]) <= 1e-5 * np.linalg.norm(want[ok])


@pytest.mark.parametrize("tag", ["da", "db", "dc", "dd"])
def test_forms_of_fewer_registers_give_the_same_bits_beside_ten_waves(tag):
    with bf.Operation(f"selftest_conv_staged_{tag}", "gemm_bf16_256x448x1792_p2") as op:
        for side, k in enumerate(op.k):
            x, w = (fill_normal(11 + 2 * side + i, int(np.prod(k.shapes[i])), 0, 1) for i in (0, 1))
            op.upload(side, *((x, w) if side == 0 else (f32_to_bf16(x), f32_to_bf16(w))))
        op.zero_outputs()
        op.launch("serial")
        want = [op.download(side).copy() for side in (0, 1)]
        op.zero_outputs()
        op.launch("bfuse", op.fused("bfuse", "_c4"))
        for side in (0, 1):
            got = op.download(side)
            assert np.any(got.view(np.uint8)) and np.array_equal(got.view(np.uint8), want[side].view(np.uint8))


@pytest.mark.parametrize("tag,s,p", [("huge_a", 4, 2), ("huge_b", 8, 1), ("huge_c", 4, 1)])
def test_images_of_two_gigabytes(tag, s, p):
    """An image of zeros but for its corners and a few other elements, each alone in its windows: every result is a product, exactly, or zero."""
    with bf.Operation(f"selftest_conv_staged_{tag}", "bias_relu_4096") as op:
        k = op.k[0]
        (_, ci, h, wd), (co, _, kh, kw), (oh, ow) = k.shapes[0], k.shapes[1], k.shapes[2][2:]
        assert ci * h * wd * 4 >= 2 ** 31
        w = fill_normal(9, co * ci * kh * kw, 0, 1).reshape(co, ci, kh, kw)
        x, want, rng = np.zeros((ci, h, wd), np.float32), np.zeros((co, oh, ow), np.float32), np.random.default_rng(3)
        places, ys = [], list(range(0, h, h // 64)) + [h - 1]
        for i, y in enumerate(ys):
            places += [(int(rng.integers(ci)), y, x0) for x0 in (0, wd // 2 + int(rng.integers(-2, 3)), wd - 1 - (y % 2 if y < h - 1 else 0))]
        places.append((ci - 1, h - 1, wd - 1 - 2 * kw))
        for c, y, x0 in places:
            x[c, y, x0] = v = np.float32(1 + rng.random())
            for oy in range(max(0, -(-(y + p - kh + 1) // s)), min(oh - 1, (y + p) // s) + 1):
                for ox in range(max(0, -(-(x0 + p - kw + 1) // s)), min(ow - 1, (x0 + p) // s) + 1):
                    assert not want[:, oy, ox].any()
                    want[:, oy, ox] = v * w[:, c, y + p - oy * s, x0 + p - ox * s]
        y = op.run_kernel(0, x, w)
        assert np.count_nonzero(want) > 1000 and np.array_equal(y.reshape(want.shape), want)
