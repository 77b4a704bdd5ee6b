"""The split-product weight gradient (lancius_amd/csrc/wgrad_split.hip): row
widths around the octets of 8 pixels, channel and tap counts at the edges of
its tiles, strides, and non-finite inputs, against fp64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import oracle
from lancius_amd import prng
from tests.conftest import case, fp32_sum_error, two_norm_error
from tests.test_gpu_gemm_split import ROUNDING

pytestmark = pytest.mark.gpu


def _run(dev, x, dy, KH, KW, stride, pad):
    N, C_in, H, W = x.shape
    _, C_out, Ho, Wo = dy.shape
    n = C_out * C_in * KH * KW
    dx, dg, do = dev.upload(x), dev.upload(dy), dev.alloc(4 * n + 4096)
    dev.fill(do, 7.0, n + 1024)
    dev.conv2d_bwd_weight(do, dg, dx, N, C_in, H, W, C_out, Ho, Wo, KH, KW, stride, pad)
    _run.kernels = dev.launched(2)
    got = dev.download(do, (n + 1024,))
    assert (got[n:] == 7.0).all()  # nothing is stored past the gradient
    for b in (dx, dg, do):
        b.free()
    return got[:n].reshape(C_out, C_in, KH, KW)


def _ref(x, dy, KH, KW, stride, pad):
    w = torch.zeros(dy.shape[1], x.shape[1], KH, KW, dtype=torch.float64, requires_grad=True)
    F.conv2d(torch.from_numpy(x).double(), w, None, stride, pad).backward(torch.from_numpy(dy).double())
    return w.grad.numpy()


def _inputs(seed, N, C_in, H, W, C_out, KH, KW, stride, pad):
    Ho, Wo = (H + 2 * pad - KH) // stride + 1, (W + 2 * pad - KW) // stride + 1
    return prng.normal(seed, (N, C_in, H, W)), prng.normal(seed + 1, (N, C_out, Ho, Wo), std=0.1)


# (N, C_in, H, W, C_out, KH, KW, stride, pad)
SHAPES = [
    (16, 64, 40, 40, 128, 3, 3, 1, 1),      # whole octets
    (9, 33, 41, 63, 72, 3, 3, 1, 1),        # rows of 63: the last octet one short
    (8, 48, 37, 65, 160, 5, 5, 1, 2),       # rows of 65: an octet of one pixel
    (6, 24, 50, 57, 130, 3, 5, 1, 2),       # an oblong filter, two channels over
    (12, 40, 45, 33, 60, 5, 5, 2, 2),       # stride 2, 64-channel tiles
    (4, 21, 35, 35, 70, 7, 7, 1, 3),
    (8, 96, 29, 31, 96, 1, 1, 1, 0),
    (8, 80, 64, 51, 144, 3, 3, 3, 0),       # stride 3
]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_wgrad_split_shapes(dev, shape):
    case(f"wgrad split {shape}")
    x, dy = _inputs(7000, *shape)
    geometry = shape[5:]
    got, ref = _run(dev, x, dy, *geometry), _ref(x, dy, *geometry)
    assert any(("wgrad_split 128x128" if shape[4] > 64 else "wgrad_split 64x128") == k for k in _run.kernels)
    assert oracle.normwise_error(got, ref) <= oracle.tolerance(dy[0, 0].size * shape[0])
    assert two_norm_error(got, ref) <= fp32_sum_error(dy[0, 0].size * shape[0])


def test_wgrad_split_is_repeatable(dev):
    shape = (9, 33, 41, 63, 72, 3, 3, 1, 1)
    x, dy = _inputs(7100, *shape)
    assert np.array_equal(_run(dev, x, dy, 3, 3, 1, 1), _run(dev, x, dy, 3, 3, 1, 1))


@pytest.mark.parametrize("stride", [1, 2])
def test_wgrad_split_non_finite(dev, stride):
    """An infinite or NaN pixel reaches the taps that see it, and no others."""
    shape = (16, 64, 41, 40, 128, 3, 3, stride, 1)
    case(f"wgrad split non-finite stride {stride}")
    x, dy = _inputs(7200, *shape)
    x[0, 3, 0, 0], x[5, 20, 17, 18] = np.inf, np.nan
    dy[7, 9, 4, 5] = -np.inf
    x[3, 50, 11, 12] = np.float32(3.4e38)  # rounds to infinity as bf16
    got, ref = _run(dev, x, dy, 3, 3, stride, 1), _ref(x, dy, 3, 3, stride, 1)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf].astype(np.float32))
    big = np.isfinite(ref) & (np.abs(ref) > 1e20)
    assert big.any()
    for part, scale in ((big, 2.0 ** -100), (np.isfinite(ref) & ~big, 1.0)):
        err = oracle.normwise_error(np.where(part, got, 0).astype(np.float64) * scale, np.where(part, ref, 0) * scale)
        assert err <= oracle.tolerance(dy[0, 0].size * 16)


@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("exponent", [0, -118, -126, -140])
def test_wgrad_split_small_operands(dev, exponent, stride):
    """x, then dY, at the low end of fp32's range, the other large enough for
    ordinary results: all 24 bits count there too."""
    shape = (16, 64, 41, 41, 128, 3, 3, stride, 1)
    case(f"wgrad split small operands 2^{exponent} stride {stride}")
    for small in ("x", "dy"):
        x, dy = _inputs(7300, *shape)
        up, down = np.float32(2.0 ** (-exponent // 3)), np.float32(2.0) ** np.float32(exponent)
        x, dy = (x * down, dy * up) if small == "x" else (x * up, dy * down)
        got = _run(dev, x, dy, 3, 3, stride, 1)
        assert any("wgrad_split" in k for k in _run.kernels), _run.kernels
        assert two_norm_error(got, _ref(x, dy, 3, 3, stride, 1)) <= fp32_sum_error(dy[0, 0].size * 16), small


@pytest.mark.parametrize("shape,kernel", [((16, 64, 41, 41, 128, 3, 3, 2, 1), "wgrad_split 128x128"),
                                          ((16, 64, 41, 40, 128, 3, 3, 1, 1), "wgrad_split 128x128"),
                                          ((12, 40, 45, 33, 60, 5, 5, 2, 2), "wgrad_split 64x128")])
def test_wgrad_split_recomputes_non_finite(dev, shape, kernel):
    """The tiles that an infinite, NaN or out-of-range value reaches are
    computed again in fp32: rows that are no whole octets, strides, both tiles."""
    case(f"wgrad split recompute {shape}")
    x, dy = _inputs(7400, *shape)
    x[0, 3, 0, 0], x[5, 20, 17, 18] = np.inf, np.nan
    dy[7, 9, -1, -1] = -np.inf
    x[3, 30, 11, 12] = np.float32(3.4e38)
    got, ref = _run(dev, x, dy, *shape[5:]), _ref(x, dy, *shape[5:])
    assert kernel in _run.kernels
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert inf.any() and np.array_equal(got[inf], ref[inf].astype(np.float32))
    big = np.isfinite(ref) & (np.abs(ref) > 1e20)
    assert big.any()
    for part, scale in ((big, 2.0 ** -100), (np.isfinite(ref) & ~big, 1.0)):
        assert two_norm_error(got[part].astype(np.float64) * scale, ref[part] * scale) <= fp32_sum_error(dy[0, 0].size * shape[0])


@pytest.mark.parametrize("images", [1, 2, 3])
def test_wgrad_few_products_round_as_fp32(dev, images):
    """A gradient over one or two pixels is one or two products an element and
    stays with the fp32 kernels."""
    x, dy = prng.normal(7500, (images, 96, 1, 1)), prng.normal(7501, (images, 160, 1, 1))
    case(f"wgrad over {images} pixels")
    got = _run(dev, x, dy, 1, 1, 1, 0)[:, :, 0, 0]
    assert "conv2d_wgrad_mfma" in _run.kernels[0]
    x, dy = x[:, :, 0, 0], dy[:, :, 0, 0]
    terms = [np.outer(dy[n].astype(np.float64), x[n].astype(np.float64)) for n in range(images)]
    ref = sum(terms)
    if images == 1:
        assert np.array_equal(got, dy.T * x)
    elif images == 2:  # both products and their sum round; a tenth for the few random numbers
        room = np.sqrt(sum(np.sum(t ** 2) for t in terms + [ref]) / np.sum(ref ** 2))
        assert two_norm_error(got, ref) <= 1.1 * ROUNDING * room
    assert two_norm_error(got, ref) <= fp32_sum_error(images)
