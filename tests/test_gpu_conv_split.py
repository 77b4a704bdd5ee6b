"""The split-product convolution (lancius_amd/csrc/conv_split.hip): channel,
pixel and tap counts at the edges of its tiles, strides, the classes of strided
input gradients, and non-finite inputs, against fp64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import oracle
from lancius_amd import ACT_NONE, ACT_RELU, prng
from tests.conftest import case, fp32_sum_error, two_norm_error
from tests.test_gpu_gemm_split import ROUNDING

pytestmark = pytest.mark.gpu


def _out(H, K, stride, pad):
    return (H + 2 * pad - K) // stride + 1


def _forward(dev, x, w, bias, stride, pad, act, packed):
    N, C_in, H, W = x.shape
    C_out, _, KH, KW = w.shape
    Ho, Wo = _out(H, KH, stride, pad), _out(W, KW, stride, pad)
    n = N * C_out * Ho * Wo
    dx, dw, do = dev.upload(x), dev.upload(w), dev.alloc(4 * n + 4096)
    db = dev.upload(bias) if bias is not None else None
    dev.fill(do, 7.0, n + 1024)
    if packed:
        pk = dev.alloc(dev.conv2d_packed_bytes(C_out, C_in, KH, KW))
        dev.conv2d_pack_weight(pk, dw, C_out, C_in, KH, KW)
        dev.conv2d_packed(do, dx, pk, db, N, C_in, H, W, C_out, KH, KW, stride, pad, act)
        _forward.kernel = dev.launched()[0]
        pk.free()
    else:
        dev.conv2d(do, dx, dw, db, N, C_in, H, W, C_out, KH, KW, stride, pad, act)
        _forward.kernel = dev.launched()[0]
    got = dev.download(do, (n + 1024,))
    assert (got[n:] == 7.0).all()  # nothing is stored past the output
    for b in (dx, dw, do, db):
        if b is not None:
            b.free()
    return got[:n].reshape(N, C_out, Ho, Wo)


def _bwd_input(dev, dy, w, H, W, stride, pad):
    N, C_out, Ho, Wo = dy.shape
    _, C_in, KH, KW = w.shape
    n = N * C_in * H * W
    dg, dw, do = dev.upload(dy), dev.upload(w), dev.alloc(4 * n + 4096)
    dev.fill(do, 7.0, n + 1024)
    dev.conv2d_bwd_input(do, dg, dw, N, C_in, H, W, C_out, Ho, Wo, KH, KW, stride, pad)
    _bwd_input.kernel = dev.launched()[0]
    got = dev.download(do, (n + 1024,))
    assert (got[n:] == 7.0).all()
    for b in (dg, dw, do):
        b.free()
    return got[:n].reshape(N, C_in, H, W)


# (N, C_in, H, W, C_out, KH, KW, stride, pad, packed, kernel: channels x pixels of a tile x groups of waves)
FORWARD = [
    (9, 64, 40, 36, 128, 3, 3, 1, 1, True, "conv2d_split 128x128 x2"),     # whole tiles, a tile a CU or less
    (40, 32, 31, 33, 132, 3, 3, 1, 1, True, "conv2d_split 128x128 x1"),    # four channels past a tile, two tiles a CU
    (24, 48, 57, 55, 96, 5, 5, 2, 2, True, "conv2d_split 128x128 x2"),     # stride 2, ragged pixels
    (64, 96, 60, 61, 128, 3, 3, 3, 0, True, "conv2d_split 128x128 x2"),    # stride 3, no padding
    (32, 37, 40, 41, 70, 3, 5, 1, 2, False, "conv2d_split 128x128 x1"),    # channels padded to 48, an oblong filter
    (8, 90, 40, 40, 200, 3, 3, 1, 1, False, "conv2d_split 128x128 x2"),    # channels padded to 96
    (10, 64, 56, 56, 64, 3, 3, 1, 1, True, "conv2d_split 64x128 x2"),      # 64-channel tiles
    (20, 64, 56, 56, 60, 3, 3, 1, 1, True, "conv2d_split 64x128 x1"),      # four channels short of one
    (10, 13, 64, 64, 51, 5, 5, 1, 2, False, "conv2d_split 64x128 x1"),     # both channel counts ragged
    (3, 48, 57, 55, 96, 5, 5, 2, 2, True, "conv2d_small 32x32"),           # few pixels of the same
    (2, 37, 40, 41, 70, 3, 5, 1, 2, False, "conv2d_small 32x32"),
    (2, 96, 30, 30, 24, 7, 7, 3, 0, False, "conv2d_small 16x16"),
    (1, 13, 64, 64, 51, 5, 5, 1, 2, False, "conv2d_small 32x32"),
]


@pytest.mark.parametrize("N,C_in,H,W,C_out,KH,KW,stride,pad,packed,kernel", FORWARD)
def test_conv_split_forward(dev, N, C_in, H, W, C_out, KH, KW, stride, pad, packed, kernel):
    case(f"conv split forward {N} {C_in}->{C_out} {H}x{W} {KH}x{KW} stride {stride}")
    x = prng.normal(6000, (N, C_in, H, W))
    w = prng.normal(6001, (C_out, C_in, KH, KW), std=float(np.sqrt(2.0 / (C_in * KH * KW))))
    b = prng.normal(6002, (C_out,))
    act = ACT_RELU if stride == 1 else ACT_NONE
    got = _forward(dev, x, w, b, stride, pad, act, packed)
    assert _forward.kernel == kernel
    ref = F.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), torch.from_numpy(b).double(), stride, pad)
    ref = (F.relu(ref) if act == ACT_RELU else ref).numpy()
    assert oracle.normwise_error(got, ref) <= oracle.tolerance(C_in * KH * KW)
    if act == ACT_NONE:  # (a ReLU of a sum near 0 keeps its error and not its size)
        assert two_norm_error(got, ref) <= fp32_sum_error(C_in * KH * KW)


# (N, C_in, H, W, C_out, KH, KW, stride, pad, kernel)
GRADIENT = [
    (8, 128, 40, 36, 128, 3, 3, 1, 1, "conv2d_split 128x128 x2"),
    (10, 160, 33, 31, 132, 5, 5, 1, 2, "conv2d_split 128x128 x2"),    # dy's channels padded to 144
    (6, 128, 57, 55, 100, 3, 3, 2, 1, "conv2d_split 128x128 x2"),     # classes of different sizes
    (24, 128, 57, 55, 72, 3, 3, 2, 1, "conv2d_split 128x128 x1"),
    (8, 64, 57, 55, 100, 3, 3, 2, 1, "conv2d_split 64x128 x2"),
    (16, 64, 57, 55, 100, 3, 3, 2, 1, "conv2d_split 64x128 x1"),
    (12, 130, 41, 43, 72, 5, 5, 2, 2, "conv2d_split 128x128 x1"),     # two channels past a tile
    (16, 96, 64, 64, 96, 1, 1, 2, 0, "conv2d_split 128x128 x1"),      # three classes without a tap
    (12, 140, 59, 61, 70, 7, 5, 3, 2, "conv2d_split 128x128 x1"),     # stride 3, an oblong filter
    (24, 64, 57, 60, 64, 3, 3, 4, 0, "conv2d_split 64x128 x1"),       # rows that no window reaches
    (8, 64, 40, 36, 128, 3, 3, 1, 1, "conv2d_direct 64x64"),          # few pixels of the same
    (2, 96, 33, 31, 48, 5, 5, 1, 2, "conv2d_small 32x32"),
    (2, 16, 78, 105, 4, 3, 3, 3, 0, "conv2d_dgrad_direct"),           # one tap of four channels an element
    (22, 16, 12, 65, 4, 3, 3, 3, 1, "conv2d_dgrad_direct"),
    (20, 2, 81, 107, 2, 7, 7, 2, 3, "conv2d_dgrad_direct"),           # two channels: no split products
    (8, 22, 90, 43, 4, 3, 3, 3, 1, "conv2d_small 32x32"),             # more pixels of the first
    (3, 40, 33, 30, 72, 3, 3, 2, 1, "conv2d_small 16x16"),
    (2, 130, 20, 23, 37, 5, 5, 2, 2, "conv2d_small 16x16"),
    (2, 24, 32, 32, 48, 1, 1, 2, 0, "conv2d_small 16x16"),
    (1, 20, 29, 31, 33, 7, 5, 3, 2, "conv2d_small 16x16"),
    (2, 16, 19, 40, 64, 3, 3, 4, 0, "conv2d_small 16x16"),
]


@pytest.mark.parametrize("N,C_in,H,W,C_out,KH,KW,stride,pad,kernel", GRADIENT)
def test_conv_split_bwd_input(dev, N, C_in, H, W, C_out, KH, KW, stride, pad, kernel):
    case(f"conv split gradient {N} {C_in}->{C_out} {H}x{W} {KH}x{KW} stride {stride}")
    Ho, Wo = _out(H, KH, stride, pad), _out(W, KW, stride, pad)
    dy = prng.normal(6100, (N, C_out, Ho, Wo))
    w = prng.normal(6101, (C_out, C_in, KH, KW), std=float(np.sqrt(2.0 / (C_out * KH * KW))))
    got = _bwd_input(dev, dy, w, H, W, stride, pad)
    assert _bwd_input.kernel == kernel
    x = torch.zeros(N, C_in, H, W, dtype=torch.float64, requires_grad=True)
    F.conv2d(x, torch.from_numpy(w).double(), None, stride, pad).backward(torch.from_numpy(dy).double())
    assert oracle.normwise_error(got, x.grad.numpy()) <= oracle.tolerance(C_out * KH * KW)
    assert two_norm_error(got, x.grad.numpy()) <= fp32_sum_error(C_out * KH * KW)


@pytest.mark.parametrize("stride", [1, 2])
def test_conv_split_non_finite(dev, stride):
    """Infinities, NaN and values above the largest bf16 reach the outputs
    whose windows hold them, with fp32's signs, and no others."""
    N, C_in, H, W, C_out = 9, 64, 40, 36, 128
    case(f"conv split non-finite stride {stride}")
    x = prng.normal(6200, (N, C_in, H, W))
    w = prng.normal(6201, (C_out, C_in, 3, 3), std=0.06)
    x[0, 3, 5, 7], x[2, 60, 20, 20] = np.inf, np.nan
    x[4, 10, 11, 12] = np.float32(3.4e38)  # rounds to infinity as bf16
    w[7, 10] *= np.float32(2.0 ** -20)
    got = _forward(dev, x, w, None, stride, 1, ACT_NONE, True)
    ref = F.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), None, stride, 1).numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf].astype(np.float32))
    big = np.isfinite(ref) & (np.abs(ref) > 1e20)
    assert big.any()
    for part, scale in ((big, 2.0 ** -100), (np.isfinite(ref) & ~big, 1.0)):
        err = oracle.normwise_error(np.where(part, got, 0).astype(np.float64) * scale, np.where(part, ref, 0) * scale)
        assert err <= oracle.tolerance(C_in * 9)


@pytest.mark.parametrize("exponent", [0, -118, -126, -140])
@pytest.mark.parametrize("what", ["forward", "gradient", "gradient, stride 2"])
def test_conv_split_small_operands(dev, what, exponent):
    """The image (or dY), then the filter, at the low end of fp32's range, the
    other large enough for ordinary results: all 24 bits count there too."""
    case(f"conv split small operands {what} 2^{exponent}")
    N, C_in, H, W, C_out = 16, 64, 56, 56, 128
    stride = 2 if "stride" in what else 1
    Ho, Wo = _out(H, 3, stride, 1), _out(W, 3, stride, 1)
    for small in ("image", "filter"):
        w = prng.normal(6301, (C_out, C_in, 3, 3))
        x = prng.normal(6300, (N, C_in, H, W) if what == "forward" else (N, C_out, Ho, Wo))
        up, down = np.float32(2.0 ** (-exponent // 3)), np.float32(2.0) ** np.float32(exponent)
        x, w = (x * down, w * up) if small == "image" else (x * up, w * down)
        x64, w64 = torch.from_numpy(x).double(), torch.from_numpy(w).double()
        if what == "forward":
            got, kernel = _forward(dev, x, w, None, 1, 1, ACT_NONE, True), _forward.kernel
            ref = F.conv2d(x64, w64, None, 1, 1)
        else:
            got, kernel = _bwd_input(dev, x, w, H, W, stride, 1), _bwd_input.kernel
            ref = F.conv_transpose2d(x64, w64, None, stride, 1, output_padding=stride - 1)
        assert "conv2d_split" in kernel, kernel
        assert two_norm_error(got, ref.numpy()) <= fp32_sum_error(9 * (C_in if what == "forward" else C_out)), small


# as FORWARD and GRADIENT, with the kernel
RECOMPUTED = [
    ("forward", 40, 32, 31, 33, 132, 3, 3, 1, 1, "conv2d_split 128x128 x1"),
    ("forward", 32, 64, 56, 56, 128, 3, 3, 2, 1, "conv2d_split 128x128 x2"),
    ("forward", 8, 90, 40, 40, 200, 3, 3, 1, 1, "conv2d_split 128x128 x2"),   # channels padded to 96
    ("forward", 10, 64, 56, 56, 64, 3, 3, 1, 1, "conv2d_split 64x128 x2"),
    ("gradient", 8, 128, 40, 36, 128, 3, 3, 1, 1, "conv2d_split 128x128 x2"),
    ("gradient", 24, 128, 57, 55, 72, 3, 3, 2, 1, "conv2d_split 128x128 x1"),
    ("gradient", 8, 64, 57, 55, 100, 3, 3, 2, 1, "conv2d_split 64x128 x2"),
]


@pytest.mark.parametrize("what,N,C_in,H,W,C_out,KH,KW,stride,pad,kernel", RECOMPUTED)
def test_conv_split_recomputes_non_finite(dev, what, N, C_in, H, W, C_out, KH, KW, stride, pad, kernel):
    """The tiles that hold infinities, NaN and values beyond the scaled range
    are computed again in fp32, in each form of the kernel."""
    case(f"conv split recompute {what} {N} {C_in}->{C_out} {H}x{W} stride {stride}")
    w = prng.normal(6401, (C_out, C_in, KH, KW), std=0.06)
    x = prng.normal(6400, (N, C_in, H, W) if what == "forward" else (N, C_out, _out(H, KH, stride, pad), _out(W, KW, stride, pad)))
    x[0, 3, 5, 7], x[2, -1, -1, -1], x[-1, 0, 0, 0] = np.inf, np.nan, -np.inf
    x[4, 10, 11, 12] = np.float32(3.4e38)
    (w[7, 10] if what == "forward" else w[10, 7])[...] *= np.float32(2.0 ** -20)
    x64, w64 = torch.from_numpy(x).double(), torch.from_numpy(w).double()
    if what == "forward":
        got, ran = _forward(dev, x, w, None, stride, pad, ACT_NONE, C_in % 16 == 0 and C_out % 4 == 0), _forward.kernel
        ref = F.conv2d(x64, w64, None, stride, pad).numpy()
    else:
        got, ran = _bwd_input(dev, x, w, H, W, stride, pad), _bwd_input.kernel
        over = ((H + 2 * pad - KH) % stride, (W + 2 * pad - KW) % stride)
        ref = F.conv_transpose2d(x64, w64, None, stride, pad, output_padding=over).numpy()
    assert ran == kernel
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert inf.any() and np.array_equal(got[inf], ref[inf].astype(np.float32))
    big = np.isfinite(ref) & (np.abs(ref) > 1e20)
    assert big.any()
    for part, scale in ((big, 2.0 ** -100), (np.isfinite(ref) & ~big, 1.0)):
        assert two_norm_error(got[part].astype(np.float64) * scale, ref[part] * scale) <= fp32_sum_error(w[0].size)


def test_conv_gradient_of_few_channels_rounds_as_fp32(dev):
    """dy of two channels at stride 2: a quarter of the elements see one tap,
    two products, and the call stays with the fp32 instructions."""
    N, C_in, C_out, H, W, stride, pad = 24, 130, 2, 64, 64, 2, 1
    case("conv gradient of two channels")
    dy = prng.normal(6700, (N, C_out, _out(H, 3, stride, pad), _out(W, 3, stride, pad)))
    w = prng.normal(6701, (C_out, C_in, 3, 3))
    got = _bwd_input(dev, dy, w, H, W, stride, pad)
    assert "conv2d_small" in _bwd_input.kernel
    centre = np.einsum("nchw,ci->nihw", dy.astype(np.float64), w[:, :, 1, 1].astype(np.float64))
    # both products and their sum round; a tenth for the few random weights
    assert two_norm_error(got[:, :, ::2, ::2], centre) <= 1.1 * ROUNDING * np.sqrt((1 + 1 + 2) / 2)
