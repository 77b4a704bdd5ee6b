"""Small products in one launch of 16 x 16 or 32 x 32 tiles
(lancius_amd/csrc/gemm_small.hip): tile and k-group edges, every operand
layout, operands at odd addresses, and non-finite values, against fp64."""
import numpy as np
import pytest

import oracle
from lancius_amd import ACT_GELU, ACT_NONE, ACT_RELU, prng
from tests.conftest import case

pytestmark = pytest.mark.gpu


def _run(dev, A, B, M, K, N, ta, tb, bias=None, act=ACT_NONE, residual=None, shift=0):
    """shift: operands start that many floats into their allocations."""
    def up(x):
        return dev.upload(np.concatenate([np.full(shift, np.nan, np.float32), np.ascontiguousarray(x).ravel()]))

    dA, dB, dC = up(A.T if ta else A), up(B.T if tb else B), dev.alloc(M * N * 4 + 4096)
    dev.fill(dC, 7.0, M * N + 1024)
    db = dev.upload(bias) if bias is not None else None
    dR = dev.upload(residual) if residual is not None else None
    dev.gemm_ex(dC, dA.ptr + 4 * shift, dB.ptr + 4 * shift, M, K, N, trans_a=ta, trans_b=tb, bias=db, act=act, residual=dR)
    _run.kernel = dev.launched()[0]
    got = dev.download(dC, (M * N + 1024,))
    assert (got[M * N:] == 7.0).all()  # nothing is stored past C
    for b in (dA, dB, dC, db, dR):
        if b is not None:
            b.free()
    return got[:M * N].reshape(M, N)


# 16 x 16 tiles with 8 and (K >= 1024) 16 waves, 32 x 32 tiles with 8 and (K >= 512) 16
SHAPES = [(1, 1, 1), (1, 7, 33), (16, 16, 16), (17, 15, 17), (33, 17, 15), (64, 10, 128), (64, 784, 128), (50, 127, 129),
          (31, 129, 48), (5, 1023, 47), (40, 1025, 33), (64, 2047, 17), (512, 512, 512), (510, 511, 513), (257, 250, 511), (255, 65, 1030)]


@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("M,K,N", SHAPES)
def test_gemm_small_shapes(dev, M, K, N, layout):
    case(f"gemm small {layout} {M}x{K}x{N}")
    ta, tb = layout[0] == "T", layout[1] == "T"
    A, B = prng.normal(2100 + M, (M, K)), prng.normal(3100 + N, (K, N))
    act = {"NN": ACT_GELU, "TN": ACT_NONE, "NT": ACT_RELU, "TT": ACT_NONE}[layout]
    bias = prng.normal(5, (N,)) if layout != "TN" else None
    R = prng.normal(6, (M, N)) if layout != "NT" else None
    got = _run(dev, A, B, M, K, N, ta, tb, bias, act, R, shift=1 if layout == "TT" else 0)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    if bias is not None:
        ref = ref + bias.astype(np.float64)
    ref = oracle.gelu(ref) if act == ACT_GELU else oracle.relu(ref) if act == ACT_RELU else ref
    if R is not None:
        ref = ref + R
    assert oracle.normwise_error(got, ref) <= oracle.tolerance(K)


@pytest.mark.parametrize("layout,small", [("TT", True), ("NT", False)])
def test_gemm_small_against_what_the_layout_can_take(dev, layout, small):
    """8080 x 2222 x 17: split products are ahead of small tiles, which are
    ahead of the fp32 kernels; with both operands transposed only the last two
    are there."""
    M, K, N = 8080, 2222, 17
    case(f"gemm small or split {layout}")
    A, B = prng.normal(2250, (M, K)), prng.normal(2251, (K, N))
    got = _run(dev, A, B, M, K, N, layout[0] == "T", True)
    assert ("gemm_f32_small" in _run.kernel) == small, _run.kernel
    assert oracle.normwise_error(got, A.astype(np.float64) @ B.astype(np.float64)) <= oracle.tolerance(K)


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_gemm_small_unaligned(dev, shift):
    case(f"gemm small operands {shift} floats off")
    A, B = prng.normal(2200, (60, 76)), prng.normal(2201, (76, 44))
    for ta, tb in ((False, False), (True, False), (False, True)):
        got = _run(dev, A, B, 60, 76, 44, ta, tb, shift=shift)
        assert oracle.normwise_error(got, A.astype(np.float64) @ B.astype(np.float64)) <= oracle.tolerance(76)


@pytest.mark.parametrize("layout", ["NN", "TN", "NT", "TT"])
def test_gemm_small_non_finite(dev, layout):
    """A load past a row's K reaches the next row: what is there stays out."""
    M, K, N = 37, 93, 41
    case(f"gemm small non-finite {layout}")
    A, B = prng.normal(2300, (M, K)), prng.normal(2301, (K, N))
    A[5, 0], A[9, 92], B[0, 7], B[92, 30] = np.inf, np.nan, -np.inf, np.inf
    got = _run(dev, A, B, M, K, N, layout[0] == "T", layout[1] == "T")
    with np.errstate(invalid="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)].astype(np.float32))
    ok = np.isfinite(ref)
    assert oracle.normwise_error(np.where(ok, got, 0), np.where(ok, ref, 0)) <= oracle.tolerance(K)
