"""Convolutions and input gradients of few pixels or channels (conv2d_small in
lancius_amd/csrc/conv_split.hip): channel and pixel counts around its 16 x 16
and 32 x 32 tiles, ragged channels, strides, and non-finite values, against
fp64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import oracle
from lancius_amd import ACT_NONE, ACT_RELU, prng
from tests.conftest import case
from tests.test_gpu_conv_split import _bwd_input, _forward

pytestmark = pytest.mark.gpu

# (N, C_in, H, W, C_out, KH, KW, stride, pad)
SHAPES = [
    (1, 16, 16, 16, 16, 3, 3, 1, 1),    # whole tiles
    (1, 3, 7, 7, 1, 3, 3, 1, 1),        # less than one tile each way
    (2, 5, 9, 13, 17, 5, 5, 1, 2),      # ragged channels both ways
    (3, 17, 8, 11, 15, 1, 1, 1, 0),
    (1, 33, 10, 10, 33, 3, 5, 1, 1),    # an oblong filter
    (32, 16, 16, 16, 32, 5, 5, 1, 2),   # 32 x 32 tiles
    (2, 31, 19, 17, 31, 7, 7, 2, 3),    # stride 2: classes of unequal pixels
    (1, 20, 16, 22, 12, 3, 3, 3, 0),    # stride 3, classes that one tap reaches
    (5, 176, 8, 9, 16, 5, 5, 1, 2),     # a long K
]
IDS = ["x".join(map(str, s)) for s in SHAPES]


def _inputs(seed, N, C_in, H, W, C_out, KH, KW, stride, pad):
    Ho, Wo = (H + 2 * pad - KH) // stride + 1, (W + 2 * pad - KW) // stride + 1
    x = prng.normal(seed, (N, C_in, H, W))
    w = prng.normal(seed + 1, (C_out, C_in, KH, KW), std=float(np.sqrt(2.0 / (C_in * KH * KW))))
    return x, w, prng.normal(seed + 2, (C_out,)), prng.normal(seed + 3, (N, C_out, Ho, Wo))


@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_conv_small_forward(dev, shape):
    case(f"conv small forward {shape}")
    x, w, b, _ = _inputs(6500, *shape)
    stride, pad = shape[7:]
    act = ACT_RELU if stride == 1 else ACT_NONE
    got = _forward(dev, x, w, b, stride, pad, act, shape[1] % 16 == 0 and shape[4] % 4 == 0)
    ref = F.conv2d(*(torch.from_numpy(a).double() for a in (x, w, b)), stride, pad).numpy()
    ref = oracle.relu(ref) if act == ACT_RELU else ref
    assert oracle.normwise_error(got, ref) <= oracle.tolerance(w[0].size)


@pytest.mark.parametrize("shape", SHAPES, ids=IDS)
def test_conv_small_input_gradient(dev, shape):
    case(f"conv small input gradient {shape}")
    x, w, _, dy = _inputs(6600, *shape)
    stride, pad = shape[7:]
    t = torch.from_numpy(x).double().requires_grad_()
    F.conv2d(t, torch.from_numpy(w).double(), None, stride, pad).backward(torch.from_numpy(dy).double())
    got = _bwd_input(dev, dy, w, *x.shape[2:], stride, pad)
    assert oracle.normwise_error(got, t.grad.numpy()) <= oracle.tolerance(w[:, 0].size)


def test_conv_small_non_finite(dev):
    """Channels are padded to 16: what the next image holds there stays out."""
    shape = (3, 5, 9, 13, 17, 3, 3, 1, 1)
    case("conv small non-finite")
    x, w, b, _ = _inputs(6700, *shape)
    x[1, 0, 0, 0], x[2, 3, 8, 12] = np.inf, np.nan
    got = _forward(dev, x, w, b, 1, 1, ACT_NONE, False)
    ref = F.conv2d(*(torch.from_numpy(a).double() for a in (x, w, b)), 1, 1).numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)].astype(np.float32))
    ok = np.isfinite(ref)
    assert oracle.normwise_error(np.where(ok, got, 0), np.where(ok, ref, 0)) <= oracle.tolerance(45)
