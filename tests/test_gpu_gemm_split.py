"""The split-product GEMM tiles (lancius_amd/csrc/gemm_split.hip): sizes at the
edges of their tiles and k-steps, each operand layout, split K, and inputs at
the ends of fp32's range, against fp64."""
import numpy as np
import pytest
import torch

import oracle
from lancius_amd import ACT_GELU, ACT_NONE, ACT_RELU, prng
from tests.conftest import case, fp32_sum_error, two_norm_error

pytestmark = pytest.mark.gpu


def _run(dev, A, B, M, K, N, ta=False, tb=False, bias=None, act=ACT_NONE, residual=None):
    dA, dB, dC = dev.upload(A), dev.upload(B), dev.alloc(M * N * 4 + 4096)
    dev.fill(dC, 7.0, M * N + 1024)
    db = dev.upload(bias) if bias is not None else None
    dR = dev.upload(residual) if residual is not None else None
    dev.gemm_ex(dC, dA, dB, M, K, N, trans_a=ta, trans_b=tb, bias=db, act=act, residual=dR)
    _run.kernels = dev.launched(2)
    got = dev.download(dC, (M * N + 1024,))
    assert (got[M * N:] == 7.0).all()  # nothing is stored past C
    for b in (dA, dB, dC, db, dR):
        if b is not None:
            b.free()
    return got[:M * N].reshape(M, N)


# 256 x 256 tiles (from 768 tiles of 128 x 128), 256 x 128, 128 x 128, and
# 128 x 128 with K split over workgroups; whole and ragged in each dimension
SHAPES = [
    (3456, 64, 3712, "256x256"),
    (3329, 16, 3847, "256x256, one k-step, ragged"),
    (3585, 35, 3585, "256x256, one row and column over"),
    (1537, 300, 2999, "256x128, ragged"),
    (2048, 257, 3071, "256x128, one k over"),
    (1024, 304, 4096, "128x128"),
    (1031, 289, 4093, "256x128, seven rows over"),
    (1153, 289, 2303, "128x128, ragged"),
    (641, 3203, 383, "128x128, split K, ragged"),
    (512, 4096, 512, "128x128, split K"),
]


@pytest.mark.parametrize("layout", ["NN", "TN", "NT"])
@pytest.mark.parametrize("M,K,N,what", SHAPES, ids=[s[-1] for s in SHAPES])
def test_gemm_split_shapes(dev, M, K, N, what, layout):
    case(f"gemm split {what} {layout} {M}x{K}x{N}")
    ta, tb = layout[0] == "T", layout[1] == "T"
    A, B = prng.normal(2000 + M, (M, K)), prng.normal(3000 + N, (K, N))
    act = {"NN": ACT_GELU, "TN": ACT_NONE, "NT": ACT_RELU}[layout]
    bias = prng.normal(5, (N,)) if layout != "TN" else None
    R = prng.normal(6, (M, N)) if layout != "NT" else None
    got = _run(dev, np.ascontiguousarray(A.T) if ta else A, np.ascontiguousarray(B.T) if tb else B, M, K, N, ta, tb,
               bias, act, R)
    assert "gemm_f32_split " + what.split(", ")[0] in _run.kernels[0 if "split K" not in what else 1]
    assert ("split K" in what) == (_run.kernels[0] == "splitk_reduce")
    ref = A.astype(np.float64) @ B.astype(np.float64)
    if bias is not None:
        ref = ref + bias.astype(np.float64)
    ref = oracle.gelu(ref) if act == ACT_GELU else oracle.relu(ref) if act == ACT_RELU else ref
    if R is not None:
        ref = ref + R
    assert oracle.normwise_error(got, ref) <= oracle.tolerance(K)
    # every row and column, the edges included
    scale = np.sqrt(np.mean(ref ** 2))
    assert np.abs(got - ref).max() <= 60 * oracle.tolerance(K) * scale


# What rounding to fp32 does to random values, two-norm (0.42 ulp / 2).  An fp32 chain of K
# products rounds the first product and each sum after it, which grow as sqrt(i):
# ROUNDING * sqrt((1 + 2 + ... + K) / K).
ROUNDING = 0.43 * 2.0 ** -24


@pytest.mark.parametrize("layout", ["NN", "TN", "NT"])
@pytest.mark.parametrize("K", [1, 2, 3, 4, 16, 33])
def test_gemm_few_products_round_as_fp32(dev, K, layout):
    """Six bf16 products leave out up to 2^-24 of each product: one or two of
    them round better with the fp32 instructions and stay there."""
    M, N = 3585, 3590
    case(f"gemm of {K} products {layout}")
    A, B = prng.normal(71, (M, K)), prng.normal(72, (K, N))
    ta, tb = layout[0] == "T", layout[1] == "T"
    got = _run(dev, np.ascontiguousarray(A.T) if ta else A, np.ascontiguousarray(B.T) if tb else B, M, K, N, ta, tb)
    assert ("gemm_f32_split" in _run.kernels[0]) == (K >= 3)
    assert two_norm_error(got, A.astype(np.float64) @ B.astype(np.float64)) <= ROUNDING * np.sqrt((K + 1) / 2)
    if K == 1:
        assert np.array_equal(got, A * B)


@pytest.mark.parametrize("layout", ["NN", "TN", "NT"])
@pytest.mark.parametrize("M,K,N", [(3585, 64, 3590), (1537, 64, 2999), (1153, 288, 2304), (512, 4096, 512)])
def test_gemm_split_keeps_its_low_products(dev, M, K, N, layout):
    """Sums of x y - h yh - h ym - m yh (h, m: the first two bf16 parts of x and
    y) leave what the parts' last products hl', mm', lh' add, 2^-17.8 rms: each of
    them is 0.55 to 0.62 of a result.  Sums of terms of 1 round at 2^-25 a step,
    2^-7 of what is left, and a tenth bounds that over the longest K here."""
    case(f"gemm split low products {layout} {M}x{K}x{N}")

    def parts(seed, shape):
        x = torch.from_numpy(prng.normal(seed, shape))
        h = x.bfloat16().float()
        return tuple(t.numpy() for t in (x, h, (x - h).bfloat16().float()))

    x, xh, xm = parts(81, (M, K // 4))
    y, yh, ym = parts(82, (K // 4, N))
    A = np.stack([x, -xh, -xh, -xm], -1).reshape(M, K)
    B = np.stack([y, yh, ym, yh], 1).reshape(K, N)
    ta, tb = layout[0] == "T", layout[1] == "T"
    got = _run(dev, np.ascontiguousarray(A.T) if ta else A, np.ascontiguousarray(B.T) if tb else B, M, K, N, ta, tb)
    assert any("gemm_f32_split" in k for k in _run.kernels)
    err = two_norm_error(got, A.astype(np.float64) @ B.astype(np.float64))
    assert err <= 0.1, err


def test_gemm_split_k_is_repeatable(dev):
    M, K, N = 512, 4096, 512
    A, B = prng.normal(1, (M, K)), prng.normal(2, (K, N))
    assert np.array_equal(_run(dev, A, B, M, K, N), _run(dev, A, B, M, K, N))


@pytest.mark.parametrize("layout", ["NN", "TN", "NT"])
@pytest.mark.parametrize("exponent", [-100, -60, 60])
def test_gemm_split_range(dev, layout, exponent):
    """Operands far from 1 keep their accuracy: the three parts have fp32's exponents."""
    M, K, N = 1024, 304, 4096
    case(f"gemm split range {layout} 2^{exponent}")
    A = prng.normal(11, (M, K)) * np.float32(2.0) ** exponent
    B = prng.normal(12, (K, N)) * np.float32(2.0) ** (-exponent // 2)
    ta, tb = layout[0] == "T", layout[1] == "T"
    got = _run(dev, np.ascontiguousarray(A.T) if ta else A, np.ascontiguousarray(B.T) if tb else B, M, K, N, ta, tb)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    assert oracle.normwise_error(got, ref) <= oracle.tolerance(K)


@pytest.mark.parametrize("layout", ["NN", "TN", "NT"])
@pytest.mark.parametrize("exponent", [0, -115, -120, -126, -140])
@pytest.mark.parametrize("M,K,N", [(1031, 289, 4093), (3456, 64, 3712), (512, 4096, 512)])
def test_gemm_split_small_operands(dev, M, K, N, exponent, layout):
    """One operand at the low end of fp32's range, subnormals included, with
    the other large enough for ordinary results: all 24 bits count there too."""
    case(f"gemm split small operands {layout} {M}x{K}x{N} 2^{exponent}")
    ta, tb = layout[0] == "T", layout[1] == "T"
    for small in "AB":
        A, B = prng.normal(13, (M, K)), prng.normal(14, (K, N))
        up, down = np.float32(2.0 ** (-exponent // 3)), np.float32(2.0) ** np.float32(exponent)
        A, B = (A * down, B * up) if small == "A" else (A * up, B * down)
        got = _run(dev, np.ascontiguousarray(A.T) if ta else A, np.ascontiguousarray(B.T) if tb else B, M, K, N, ta, tb)
        assert any("gemm_f32_split" in k for k in _run.kernels)
        assert two_norm_error(got, A.astype(np.float64) @ B.astype(np.float64)) <= fp32_sum_error(K), small


@pytest.mark.parametrize("layout", ["NN", "TN", "NT"])
@pytest.mark.parametrize("M,K,N", [(1031, 289, 4093), (3456, 64, 3712), (512, 4096, 512), (1153, 289, 2303)])
def test_gemm_split_non_finite(dev, M, K, N, layout):
    """Infinities, NaN and values above the largest bf16 give what fp32
    arithmetic gives: an infinite input spoils its own row or column only,
    with the sign of its products, and everything else keeps its value."""
    case(f"gemm split non-finite {layout} {M}x{K}x{N}")
    A, B = prng.normal(21, (M, K)), prng.normal(22, (K, N))
    A[3, 5], A[M - 1, K - 1] = np.inf, np.nan
    B[7 % K, 9] = -np.inf
    A[40, 2] = np.finfo(np.float32).max  # rounds to infinity as bf16
    B[2, :] *= np.float32(2.0 ** -30)
    ta, tb = layout[0] == "T", layout[1] == "T"
    got = _run(dev, np.ascontiguousarray(A.T) if ta else A, np.ascontiguousarray(B.T) if tb else B, M, K, N, ta, tb)
    with np.errstate(all="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf].astype(np.float32))
    ok = np.isfinite(ref)
    rows = np.flatnonzero(ok.any(axis=1) & (np.arange(M) != 40))
    keep = ok[rows]
    assert oracle.normwise_error(np.where(keep, got[rows], 0.0), np.where(keep, ref[rows], 0.0)) <= oracle.tolerance(K)
    big = ok[40]
    assert oracle.normwise_error(got[40, big].astype(np.float64) * 2.0 ** -100, ref[40, big] * 2.0 ** -100) <= oracle.tolerance(K)


def test_gemm_split_grouped(dev):
    """Groups share a launch: each keeps its own operands, bias and residual."""
    n, M, K, N = 3, 700, 520, 900
    case("gemm split grouped")
    As = [prng.normal(31 + i, (M, K)) for i in range(n)]
    Bs = [prng.normal(41 + i, (K, N)) for i in range(n)]
    bias = [prng.normal(51 + i, (N,)) for i in range(n)]
    Rs = [prng.normal(61 + i, (M, N)) for i in range(n)]
    up = [[dev.upload(x) for x in xs] for xs in (As, Bs, bias, Rs)]
    Cs = [dev.alloc(M * N * 4) for _ in range(n)]
    dev.gemm_grouped(Cs, up[0], up[1], M, K, N, up[2], ACT_RELU, up[3])
    for i in range(n):
        ref = oracle.relu(As[i].astype(np.float64) @ Bs[i].astype(np.float64) + bias[i]) + Rs[i]
        assert oracle.normwise_error(dev.download(Cs[i], (M, N)), ref) <= oracle.tolerance(K)
    for b in Cs + [x for xs in up for x in xs]:
        b.free()
