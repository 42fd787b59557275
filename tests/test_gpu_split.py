"""fp32 products on the bf16 matrix cores (csrc/split.h, ops_gemm_split.h, ops_gemm_splitk.h): the edges of tiles and stages against the oracle
(products: numpy in double), alone and fused; their error against 64 bits; and operands that three bf16 cannot hold."""
import numpy as np
import pytest
import torch

import bfuse_project_amd as bf
from bfuse_project_amd import patterns
from bfuse_project_amd.operation import fill_normal
from oracle import oracle as orf
from tests.test_gpu_conv_tile import _check

pytestmark = pytest.mark.gpu


def _product(a, b):
    """[M, K] . [K, N], or [b, M, K] . [b, N, K]^T"""
    a, b = a.astype(np.float64), b.astype(np.float64)
    return a[..., 0, 0] @ b[..., 0, 0] if a.shape[2] == 1 else np.matmul(a[..., 0], b[..., 0].transpose(0, 2, 1))


@pytest.mark.parametrize("tag,partner,kind,suffix", [
    ("a", "layernorm_8x256", "bfuse", "_c4"), ("b", "bias_relu_4096", None, ""), ("c", "bias_relu_4096", None, ""), ("d", "bias_relu_4096", None, ""),
    ("e", "bias_relu_4096", "hfuse", ""), ("f", "conv3x3_f32_32x12x12_32", "hfuse", ""), ("m", "bias_relu_4096", None, ""), ("n", "bias_relu_4096", None, ""),
    ("o", "bias_relu_4096", None, ""), ("p", "bias_relu_4096", None, ""), ("q", "bias_relu_4096", None, "")])
def test_split_product_against_numpy_and_fused(tag, partner, kind, suffix):
    _check(f"selftest_gemm_split_{tag}", lambda a, b: _product(a, b).astype(np.float32), partner, kind, suffix)


def _gelu(x):
    return 0.5 * x * (1 + np.tanh(0.797885 * (x + 0.044715 * x ** 3)))


@pytest.mark.parametrize("tag,partner,kind,suffix", [
    ("a", "layernorm_8x256", "bfuse", "_c4"), ("b", "bias_relu_4096", "hfuse", ""), ("b", "conv3x3_f32_32x12x12_32", "hfuse", ""), ("c", "bias_relu_4096", None, ""),
    ("d", "bias_relu_4096", None, ""), ("e", "bias_relu_4096", None, "")])
def test_split_k_product_against_numpy_and_fused(tag, partner, kind, suffix):
    _check(f"selftest_gemm_splitk_{tag}", lambda a, b: (_gelu if tag == "a" else np.asarray)(_product(a, b)).astype(np.float32), partner, kind, suffix)


@pytest.mark.parametrize("tag,s,partner,kind,suffix", [("g", 1, "bias_relu_4096", None, ""), ("h", 2, "bias_relu_4096", None, ""), ("r", 1, "layernorm_8x256", "bfuse", "_c4")])
def test_split_1x1_convolution_against_the_oracle(tag, s, partner, kind, suffix):
    _check(f"selftest_gemm_split_{tag}", lambda x, w: orf.conv2d(x, w, s=s, p=0), partner, kind, suffix)


@pytest.mark.parametrize("tag,s,p", [("i", 1, 1), ("j", 2, 0), ("k", 1, 2), ("l", 3, 2)])
def test_split_convolution_against_the_oracle(tag, s, p):
    _check(f"selftest_gemm_split_{tag}", lambda x, w: orf.conv2d(x, w, s=s, p=p), "bias_relu_4096", None, "")


@pytest.mark.parametrize("tag,s,p", [("i", 1, 1), ("j", 2, 0)])
@pytest.mark.parametrize("scale", [2.0 ** -118, 2.0 ** -140])
def test_infinite_and_tiny_pixels_of_a_split_convolution(tag, s, p, scale):
    """An infinite, a NaN and a lowest value are in the windows that hold them and in no others (padding beside them is not
    multiplied), an image of values below bf16's bits keeps its own."""
    name = f"selftest_gemm_split_{tag}"
    x, w = _operands(name)
    w = np.abs(w) + np.float32(0.5)
    x[0, 3, 0, 0], x[1, 5, 4, 3], x[1, 2, 0, 6], x[0, 7, 5, 5] = np.inf, np.nan, -np.inf, np.finfo(np.float32).min
    x[2] *= np.float32(scale)
    w *= np.float32(2.0 ** 60)
    with np.errstate(all="ignore"):
        want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), stride=s, padding=p).numpy()
        f = want.astype(np.float32)
    y = _run(name, x, w)
    assert np.array_equal(np.isnan(y), np.isnan(f)) and np.array_equal(np.isposinf(y), np.isposinf(f)) and np.array_equal(np.isneginf(y), np.isneginf(f))
    for n in range(x.shape[0]):
        ok = np.isfinite(f[n])
        assert ok.any() and np.linalg.norm((y[n][ok] - want[n][ok])) <= 1e-5 * np.linalg.norm(want[n][ok])


def _run(name, x, w):
    with bf.Operation(name, "bias_relu_4096") as op:
        op.upload(0, x, w)
        op.zero_outputs()
        op.launch("kernel1")
        return op.download(0).reshape(op.k[0].shapes[2])


def _operands(name):
    with bf.Operation(name, "bias_relu_4096") as op:
        k = op.k[0]
    return [fill_normal(11 + i, int(np.prod(k.shapes[i])), 0, 1).reshape(k.shapes[i]) for i in (0, 1)]


@pytest.mark.parametrize("tag,steps,groups", [("_d", 4096 // 32, 1), ("_m", 256 // 32, 1), ("_b", 256 // 32, 2)])
def test_split_product_is_closer_to_64_bits_than_one_fp32_sum(tag, steps, groups):
    """A sum rounded r times on its way is off by at most u = 2^-24 of what it has grown to each time, u sqrt(r / 2) (2-norm).  A group
    adds a partial sum every four steps of 32 k, r = steps / 4; those are rounded six times a step on sums of half of four steps,
    24 steps / groups times 2 / (steps / groups) of the whole: 12 u^2 more.  The products left out add less than u / 2, adding
    the groups u."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    want = _product(x, w)
    err = np.linalg.norm(_run(name, x, w).reshape(want.shape) - want) / np.linalg.norm(want)
    assert err <= 2.0 ** -24 * ((steps / groups / 8 + 12) ** 0.5 + 0.5 + (groups > 1))


@pytest.mark.parametrize("tag,steps,groups", [("k_b", 6 * 192 // 32, 2), ("k_c", 6 * 128 // 32, 4), ("k_d", 6 * 192 // 32, 2), ("k_e", 6 * 256 // 32, 4)])
def test_split_k_product_is_closer_to_64_bits_than_one_fp32_sum(tag, steps, groups):
    """One sum a wave, rounded six times for 32 k, `groups` of which are added."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    want = _product(x, w)
    err = np.linalg.norm(_run(name, x, w).reshape(want.shape) - want) / np.linalg.norm(want)
    assert err <= 2.0 ** -24 * ((steps / 2 / groups) ** 0.5 + 0.5 + (groups > 1))


@pytest.mark.parametrize("tag", ["_a", "_b", "_e", "k_b", "k_c", "k_d", "k_e"])
@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -118, 2.0 ** 100])
def test_scaled_operands_keep_their_bits(tag, scale):
    """A power of two on an operand is one on the result, however small the operand's own low bits become (whole operand, one
    row or column among others, a column of zeros beside it)."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    scale = np.float32(scale)
    u = 2.0 ** -24 * x.shape[1] ** 0.5 * 2     # twice the bound of one sum rounded after every product
    want = _product(x, w)
    for a, b, f in ((x * scale, w, scale), (x, w * scale, scale)):
        y = _run(name, a, b).reshape(want.shape).astype(np.float64) / float(f)
        assert np.linalg.norm(y - want) <= u * np.linalg.norm(want)
    a, rows = x.copy().reshape(-1, x.shape[-3] if x.shape[2] == 1 else x.shape[-2]), slice(3, None, 16)
    a[rows] *= scale
    a[5] = 0
    a = a.reshape(x.shape)
    want = _product(a, w)
    y = _run(name, a, w).reshape(want.shape).astype(np.float64)
    want, y = want.reshape(-1, want.shape[-1]), y.reshape(-1, want.shape[-1])
    for r in range(want.shape[0]):
        assert np.linalg.norm(y[r] - want[r]) <= u * np.linalg.norm(want[r]), r


@pytest.mark.parametrize("tag", ["_a", "_b", "_e", "k_b", "k_c", "k_d", "k_e"])
@pytest.mark.parametrize("scale", [2.0 ** -112, 2.0 ** -125, 2.0 ** -136, 2.0 ** -145])
def test_values_with_bits_below_the_parts_keep_them(tag, scale):
    """Operands, or some rows of them, of which one bf16 part or all three are zero or hold less than the value (results are
    ordinary numbers: the other operand is that much larger)."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    u = 2.0 ** -24 * x.shape[1 if x.shape[2] == 1 else 2] ** 0.5 * 2     # as above
    big = np.float32(2.0 ** 90)
    some = x.copy().reshape(-1, x.shape[-3] if x.shape[2] == 1 else x.shape[-2])
    some[3::16] *= np.float32(scale)
    for a, b in ((x * np.float32(scale), w * big), (x * big, w * np.float32(scale)), (some.reshape(x.shape), w * big)):
        want = _product(a, b)
        y = _run(name, a, b).reshape(want.shape).astype(np.float64)
        want, y = want.reshape(-1, want.shape[-1]), y.reshape(-1, want.shape[-1])
        for r in range(want.shape[0]):
            assert np.linalg.norm(y[r] - want[r]) <= u * np.linalg.norm(want[r]), r


def _one_hot(name, x, w, side, values):
    """The operands with `side` replaced by one value a row (column) of the result, at k = row (column) modulo K, and what the
    product then is: that value times the other operand's k."""
    rows = x.shape[2] == 1                         # [M, K] . [K, N], or [b, M, K] . [b, N, K]^T
    x, w = x.copy(), w.copy()
    if side == 0:
        x[...] = 0
        m = x.shape[0 if rows else 1]
        k = np.arange(m) % x.shape[1 if rows else 2]
        if rows:
            x[np.arange(m), k, 0, 0] = values[:m]
        else:
            x[:, np.arange(m), k, 0] = values[:m]
    else:
        w[...] = 0
        n = w.shape[1]
        k = np.arange(n) % w.shape[0 if rows else 2]
        if rows:
            w[k, np.arange(n), 0, 0] = values[:n]
        else:
            w[:, np.arange(n), k, 0] = values[:n]
    return x, w, _product(x, w)


@pytest.mark.parametrize("tag", ["_a", "_b", "_e", "k_b", "k_c", "k_d", "k_e"])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -112, 2.0 ** -120, 2.0 ** -126])
@pytest.mark.parametrize("side", [0, 1])
def test_a_product_with_a_permutation_is_exact(tag, scale, side):
    """... whatever small values lie beside ordinary ones."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    (w if side == 0 else x).reshape(-1)[3::7] *= np.float32(scale)
    x, w, want = _one_hot(name, x, w, side, np.ones(max(x.size, w.size), np.float32))
    assert np.array_equal(_run(name, x, w).reshape(want.shape), want.astype(np.float32))


@pytest.mark.parametrize("tag", ["_a", "_b", "_e", "k_b", "k_c", "k_d", "k_e"])
@pytest.mark.parametrize("side", [0, 1])
def test_sums_of_one_product(tag, side):
    """One product of two values of 24 bits.  With u = 2^-24, of the product: its sum is rounded (u), after what the smaller partial
    products came to has been cut off at half a unit of its last place (u); the two larger ones of the partial products that are
    left out are u / 2 each at most; the five smaller ones, 2^-7 of the product together, are cut and rounded on their way."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    # the worst is near 1 + 2^-8, where the second part is half a bit of the first
    near = fill_normal(5, x.size + w.size, 0, 1)
    worst = (np.float32(1) + np.float32(2.0 ** -8) + np.arange(w.size + x.size, dtype=np.float32) % 512 * np.float32(2.0 ** -20)).astype(np.float32)
    for values, other in ((near, near), (worst, worst)):
        a, b = (x, other[: w.size].reshape(w.shape)) if side == 0 else (other[: x.size].reshape(x.shape), w)
        a, b, want = _one_hot(name, a, b, side, values)
        y = _run(name, a, b).reshape(want.shape)
        assert np.all(np.abs(y - want) <= 2.0 ** -24 * (3 + 10 * 2.0 ** -7) * np.abs(want))


@pytest.mark.parametrize("tag,partner,kind,suffix", [
    ("_a", "layernorm_8x256", "bfuse", "_c4"), ("_e", "bias_relu_4096", "hfuse", ""), ("_f", "conv3x3_f32_32x12x12_32", "hfuse", ""),
    ("k_a", "layernorm_8x256", "bfuse", "_c4"), ("k_b", "bias_relu_4096", "hfuse", ""), ("k_b", "conv3x3_f32_32x12x12_32", "hfuse", "")])
@pytest.mark.parametrize("value", [2.0 ** -120 * 1.2345678, np.inf])
def test_fused_kernels_multiply_again_where_the_parts_do_not_do(tag, partner, kind, suffix, value):
    """One value that its parts do not hold: the tiles it is in are done again, with as many barriers as that takes, and fused
    results are the unfused ones' bits."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    x.reshape(-1)[x.shape[1 if x.shape[2] == 1 else 2] + 2] = value
    with bf.Operation(name, partner) as op:
        P = [fill_normal(21 + i, int(np.prod(op.k[1].shapes[i])), 0, 1) for i in (0, 1)]
        o1, o2 = op.run_kernel(0, x, w), op.run_kernel(1, *P)
        f1, f2 = op.run_fuse(op.fused(kind, suffix), x, w, *P)
    with np.errstate(all="ignore"):
        want = (_gelu if tag == "k_a" else np.asarray)(_product(x, w))
    o = o1.reshape(want.shape)
    ok = np.isfinite(want)
    assert np.array_equal(np.isfinite(o), ok) and np.linalg.norm(o[ok] - want[ok]) <= 1e-5 * np.linalg.norm(want[ok])
    assert np.array_equal(o1.view(np.uint32), f1.view(np.uint32)) and np.array_equal(o2.view(np.uint32), f2.view(np.uint32))


@pytest.mark.parametrize("side,value", [(0, 2.0 ** -120 * 1.2345678), (1, 2.0 ** -120 * 1.2345678), (0, np.inf), (1, np.inf)])
def test_the_form_of_half_the_waves_does_the_same_results_again(side, value):
    """Ten waves of 16 rows alone, five of 32 in the fused kernel: one image's pixel or one channel's weight that the parts do not hold."""
    x, w = _operands("selftest_gemm_split_r")
    (x, w)[side][(1, 5, 4, 3) if side == 0 else (19, 7, 0, 0)] = value
    with bf.Operation("selftest_gemm_split_r", "layernorm_8x256") as op:
        assert op.k[0].block[0] == 640 and op.fused("bfuse", "_c4").block[0] == 320
        P = [fill_normal(21 + i, int(np.prod(op.k[1].shapes[i])), 0, 1) for i in (0, 1)]
        o = op.run_kernel(0, x, w)
        f = op.run_fuse(op.fused("bfuse", "_c4"), x, w, *P)[0]
    assert np.isfinite(o).all() == np.isfinite(value) and np.isfinite(o).any()
    assert np.array_equal(o.view(np.uint32), f.view(np.uint32))


@pytest.mark.parametrize("tag,side,at,kept", [("_a", 0, 150, 128), ("_f", 0, 200, 112), ("_e", 1, 79, 64)])
def test_overlapping_tiles_leave_their_neighbours_results_to_them(tag, side, at, kept):
    """A value that its parts do not hold in the last row (column) tile: that one is done again, and the rows (columns) before
    the last tile's own keep their bits."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    k = np.s_[at, 2] if x.shape[2] == 1 else np.s_[:, at, 2]
    out = []
    for v in (0, 2.0 ** -120 * 1.2345678):
        (x, w)[side][k] = v
        out.append(_run(name, x, w).reshape(_product(x, w).shape))
    a, b = (o[..., :kept, :] if side == 0 else o[..., :kept] for o in out)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    assert not np.array_equal(out[0], out[1])


@pytest.mark.parametrize("tag", ["_a", "_b", "_e", "k_b", "k_c", "k_d", "k_e"])
def test_infinities_nan_and_the_largest_values(tag):
    """What does not fit three bf16 gives what fp32 arithmetic gives: infinite where it is, NaN where it is, finite elsewhere."""
    name = f"selftest_gemm_split{tag}"
    x, w = _operands(name)
    x2 = x.reshape(-1, x.shape[1] if x.shape[2] == 1 else x.shape[2])      # rows
    big = np.float32(3.4e38)
    w = np.abs(w) + np.float32(0.5)
    x2[2, 1], x2[4, 0], x2[4, 1], x2[7, 3] = np.inf, np.inf, -np.inf, np.nan
    x2[9] = 0
    x2[9, 2], x2[11, 4] = np.finfo(np.float32).min, big
    if tag != "_e":
        w2 = w.reshape(w.shape[0], w.shape[1])
        w2[2] = np.float32(0.5)                                            # 0.5 * the lowest value stays finite
        w2[1, 5], w2[0, 6] = np.inf, np.nan
    with np.errstate(all="ignore"):
        want = _product(x, w).astype(np.float32).reshape(-1, _product(x, w).shape[-1])
    y = _run(name, x, w).reshape(want.shape)
    assert np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(np.isposinf(y), np.isposinf(want)) and np.array_equal(np.isneginf(y), np.isneginf(want))
    ok = np.isfinite(want)
    assert ok.any() and np.all(np.abs(y[ok] - want[ok]) <= 1e-5 * np.maximum(np.abs(want[ok]), np.sqrt(np.float32(x2.shape[1]))))


CONV_PATCHES = [("a", 1), ("b", 1), ("c", 0), ("d", 1), ("e", 0), ("f", 2), ("g", 1), ("h", 1)]


@pytest.mark.parametrize("tag,p", CONV_PATCHES)
def test_convolution_from_a_patch_against_the_oracle_and_fused(tag, p):
    partner, kind, suffix = {"a": ("layernorm_8x256", "bfuse", "_c4"), "b": ("bias_relu_4096", "hfuse", ""),
                             "d": ("conv3x3_f32_32x12x12_32", "hfuse", "")}.get(tag, ("bias_relu_4096", None, ""))
    _check(f"selftest_conv_split_{tag}", lambda x, w: orf.conv2d(x, w, s=1, p=p), partner, kind, suffix)


@pytest.mark.parametrize("tag,p", CONV_PATCHES)
@pytest.mark.parametrize("where", ["image", "filter"])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -118, 2.0 ** -140])
def test_values_that_parts_do_not_hold_in_a_patch_or_its_filters(tag, p, where, scale):
    """Infinite, NaN and lowest values are in the results that have them in their window (padding and places beside an image
    are not multiplied), and values below bf16's bits keep theirs: what fp32 arithmetic gives."""
    _values_that_parts_do_not_hold(f"selftest_conv_split_{tag}", 1, p, where, scale)


def _values_that_parts_do_not_hold(name, s, p, where, scale):
    x, w = _operands(name)
    w = np.abs(w) + np.float32(0.5)
    if where == "image":
        x[0, 3, 0, 0], x[1, 5, 4, 3], x[-1, 2, 0, 4], x[0, 7, 4, 4] = np.inf, np.nan, -np.inf, np.finfo(np.float32).min
        x[1] *= np.float32(scale)
    else:
        x = np.abs(x) + np.float32(0.5)
        w[17, 3, 1, 1], w[1, 5, 0, 2], w[-1, 2, 2, 0] = np.inf, np.nan, np.finfo(np.float32).min
        w[2] *= np.float32(scale)
    (w if where == "image" else x)[...] *= np.float32(2.0 ** 60)
    with np.errstate(all="ignore"):
        want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), stride=s, padding=p).numpy()
        f = want.astype(np.float32)
    y = _run(name, x, w)
    assert np.array_equal(np.isnan(y), np.isnan(f)) and np.array_equal(np.isposinf(y), np.isposinf(f)) and np.array_equal(np.isneginf(y), np.isneginf(f))
    u = 2.0 ** -24 * np.prod(w.shape[1:]) ** 0.5 * 2     # twice the bound of one sum rounded after every product
    for part in [(n, slice(None)) for n in range(x.shape[0])] + [(slice(None), m) for m in range(w.shape[0])]:
        ok = np.isfinite(f[part]) & (np.abs(want[part]) < 2.0 ** 120)      # (the lowest value's products drown the others)
        assert np.linalg.norm(y[part][ok] - want[part][ok]) <= u * np.linalg.norm(want[part][ok])


@pytest.mark.parametrize("tag,channels", [("a", 64), ("c", 96), ("e", 128), ("g", 96), ("h", 160)])
def test_convolution_from_a_patch_is_closer_to_64_bits_than_one_fp32_sum(tag, channels):
    """As the products: partial sums of n taps of 32 channels are each rounded 6 n times while they grow, and added once; n is two,
    or three where more than 128 channels are."""
    name = f"selftest_conv_split_{tag}"
    x, w = _operands(name)
    p = dict(CONV_PATCHES)[tag]
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), padding=p).numpy()
    err = np.linalg.norm(_run(name, x, w) - want) / np.linalg.norm(want)
    steps = channels // 32 * 9
    assert err <= 2.0 ** -24 * ((steps / 4 + 9) ** 0.5 + 0.5)


@pytest.mark.parametrize("tag", ["b", "d"])
def test_a_convolution_from_a_patch_of_32_channels_adds_up_every_tap(tag):
    """Nine partial sums, added up: 9 / 2 roundings of the whole in all; each of them rounded six times while it grows, 6 / 2 of a ninth
    (2-norms squared): 9 * 3 / 9 more.  A rounding is off by u / sqrt(3), evenly spread over half a unit of the last place.  (Sums of two taps
    are off by 1.6 - 1.7 u.)"""
    name = f"selftest_conv_split_{tag}"
    x, w = _operands(name)
    want = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), padding=dict(CONV_PATCHES)[tag]).numpy()
    err = np.linalg.norm(_run(name, x, w) - want) / np.linalg.norm(want)
    assert err <= 2.0 ** -24 * ((4.5 + 3) / 3) ** 0.5


def test_filters_are_taken_apart_for_every_launch_and_side():
    """The parts are the launch's own filters': new ones, two sides at once on two streams, replays of a graph, a plan at run time."""
    name = "selftest_conv_split_a"
    with bf.Operation(name, name) as op:
        k = op.k[0]
        X = [fill_normal(31 + i, int(np.prod(k.shapes[0])), 0, 1) for i in range(2)]
        W = [fill_normal(41 + i, int(np.prod(k.shapes[1])), 0, 1) for i in range(2)]
        want = [[op.run_kernel(0, x, w) for w in W] for x in X]
        assert np.array_equal(op.run_kernel(0, X[0], W[0]), want[0][0])
        for a, b in ((0, 1), (1, 0)):
            y0, y1 = op.run_parallel(X[0], W[a], X[1], W[b])
            assert np.array_equal(y0, want[0][a]) and np.array_equal(y1, want[1][b])
        for rnd in range(3):
            op.upload(0, X[0], W[rnd % 2])
            op.upload(1, X[1], W[1])
            for mode in ("parallel", "serial", "kernel1"):
                op.zero_outputs()
                assert op.time_graph(mode, chain=2, reps=2) > 0
                assert np.array_equal(op.download(0), want[0][rnd % 2]) and (mode == "kernel1" or np.array_equal(op.download(1), want[1][1]))
                assert (op.time(mode, warmup=1, reps=2)[0] > 0).all()
        P = [fill_normal(21 + i, 8 * 256 if i == 0 else 512, 0, 1) for i in (0, 1)]
    with bf.Operation(name, "layernorm_8x256") as op:
        for w in (0, 1):
            assert np.array_equal(op.run_fuse(op.fused("bfuse", "_c4"), X[0], W[w], *P)[0], want[0][w])
    with bf.Operation("selftest_conv_split_f", "layernorm_8x256") as op:
        k = op.k[0]
        x, W = fill_normal(31, int(np.prod(k.shapes[0])), 0, 1), [fill_normal(41 + i, int(np.prod(k.shapes[1])), 0, 1) for i in range(2)]
        dims = [patterns.LaunchDims(tuple(q.grid), tuple(q.block)) for q in op.k]
        rt = op.set_plan(op.fused_rt(), patterns.plan_blocks("ranges", dims), 2)
        for w in W:
            y = op.run_kernel(0, x, w)
            assert np.array_equal(op.run_fuse(rt, x, w, *P)[0], y)


@pytest.mark.parametrize("tag,side,value", [(tag, side, value) for tag in ("a", "b", "h", "i", "j", "l", "r", "s") for side in (0, 1)
                                            for value in (1.0, 2.0 ** -120 * 1.2345678, np.inf) if tag != "l" or value == 1.0])
def test_an_operand_taken_apart_before_gives_the_same_bits(tag, side, value):
    """The same products of the same parts, whatever values lie in either operand (l: tiles of 112 columns for 64; those with
    a value that its parts do not hold are done again, so that one compares its ordinary operands alone; the others are the next test's)."""
    x, w = _operands(f"selftest_gemm_split_{tag}")
    (x, w)[side].reshape(-1)[[7, 1001]] = value
    with bf.Operation(f"selftest_gemm_split_{tag}", f"selftest_gemm_split_{tag}_p") as op:
        for i in (0, 1):
            op.upload(i, x, w)
        op.zero_outputs()
        op.launch("serial")
        a, b = op.download(0), op.download(1)
    assert np.isfinite(a).any() and np.array_equal(a.view(np.uint32), b.view(np.uint32))
    if tag == "r":
        with bf.Operation("selftest_gemm_split_r_p", "layernorm_8x256") as op:
            P = [fill_normal(21 + i, int(np.prod(op.k[1].shapes[i])), 0, 1) for i in (0, 1)]
            assert np.array_equal(op.run_fuse(op.fused("bfuse", "_c4"), x, w, *P)[0].view(np.uint32), a.view(np.uint32))


@pytest.mark.parametrize("where", ["image", "filter"])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -118, 2.0 ** -140])
def test_values_that_parts_do_not_hold_in_filters_of_30_taps_taken_apart_before(where, scale):
    _values_that_parts_do_not_hold("selftest_gemm_split_l_p", 3, 2, where, scale)


def test_a_fused_kernel_of_two_operators_whose_operands_are_taken_apart():
    a, b = "selftest_conv_split_a", "selftest_gemm_split_r_p"
    with bf.Operation(a, b) as op:
        X = [fill_normal(51 + i, int(np.prod(k.shapes[0])), 0, 1) for i, k in enumerate(op.k)]
        for seed in (61, 71):                          # new filters with every launch
            W = [fill_normal(seed + i, int(np.prod(k.shapes[1])), 0, 1) for i, k in enumerate(op.k)]
            want = [op.run_kernel(i, X[i], W[i]) for i in (0, 1)]
            got = op.run_fuse(op.fused("bfuse", "_c4"), X[0], W[0], X[1], W[1])
            assert all(np.array_equal(g.view(np.uint32), w.view(np.uint32)) for g, w in zip(got, want))


@pytest.mark.parametrize("tag", ["a", "b", "d"])
@pytest.mark.parametrize("value", [1.0, 2.0 ** -120 * 1.2345678, np.inf])
def test_a_patch_convolution_of_twice_the_waves_gives_the_same_bits(tag, value):
    """Slim, beside ten waves: whatever values lie in either operand."""
    name = f"selftest_conv_split_{tag}"
    x, w = _operands(name)
    with bf.Operation(name, "gemm_bf16_256x448x1792_p2") as op:
        q = [fill_normal(81 + i, int(np.prod(op.k[1].shapes[i])), 0, 1) for i in (0, 1)]
        q = [bf.operation.f32_to_bf16(v) for v in q]
        for side in (0, 1):
            a, b = x.copy(), w.copy()
            (a, b)[side].reshape(-1)[[7, 1001]] = value
            want = op.run_kernel(0, a, b), op.run_kernel(1, *q)
            got = op.run_fuse(op.fused("bfuse", "_c4"), a, b, *q)
            assert np.isfinite(want[0]).any()
            assert np.array_equal(got[0].view(np.uint32), want[0].view(np.uint32)) and np.array_equal(got[1].view(np.uint16), want[1].view(np.uint16))


@pytest.mark.parametrize("tag", ["a", "b", "c", "d"])
@pytest.mark.parametrize("value", [1.0, 2.0 ** -120 * 1.2345678, np.inf])
@pytest.mark.parametrize("side", [0, 1])
def test_results_in_whole_lines_are_the_same_bits(tag, value, side):
    """... also those that are done again where three parts do not hold an operand, of an ordinary one, one tiny row or column among others and one infinity, alone and fused."""
    name = f"selftest_gemm_lines_{tag}"
    ops = _operands(name)
    ops[side].reshape(ops[side].shape[0], -1)[-1, 5::7] *= np.float32(value)
    want = _run(name, *ops)
    assert np.any(want) and np.array_equal(_run(name + "_w", *ops).view(np.uint32), want.view(np.uint32))
    if tag in "ad":
        with bf.Operation(name + "_w", "layernorm_8x256") as op:
            op.upload(0, *ops)
            op.upload(1, *(fill_normal(21 + i, int(np.prod(op.k[1].shapes[i])), 0, 1) for i in (0, 1)))
            op.zero_outputs()
            op.launch("bfuse", op.fused("bfuse", "_c4"))
            assert np.array_equal(op.download(0).view(np.uint32).ravel(), want.view(np.uint32).ravel())
