"""The split-product attention kernel (lancius_amd/csrc/attention_split.hip):
ragged query and key counts at the edges of its tiles, each head dim, both
grids (one tile per CU, and more), and non-finite inputs, against fp64."""
import numpy as np
import pytest

import oracle
from lancius_amd import prng
from tests.conftest import case, fp32_sum_error, two_norm_error

pytestmark = pytest.mark.gpu


def _run(dev, q, k, v, causal):
    B, Sq, Hq, D = q.shape
    Skv, Hkv = k.shape[1], k.shape[2]
    dq, dk, dv, do = dev.upload(q), dev.upload(k), dev.upload(v), dev.alloc(q.nbytes + 1024)
    dev.fill(do, 7.0, q.size + 256)
    dev.attention_gqa(do, dq, dk, dv, B, Sq, Skv, Hq, Hkv, D, causal)
    _run.kernel = dev.launched()[0]
    got = dev.download(do, (q.size + 256,))
    assert (got[q.size:] == 7.0).all()  # nothing is stored past the output
    for b in (dq, dk, dv, do):
        b.free()
    return got[:q.size].reshape(q.shape)


def _ref(q, k, v, causal):
    B, Sq, Hq, D = q.shape
    Skv, group = k.shape[1], Hq // k.shape[2]
    out = np.empty(q.shape)
    with np.errstate(all="ignore"):
        for b in range(B):
            for h in range(Hq):
                s = q[b, :, h].astype(np.float64) @ k[b, :, h // group].astype(np.float64).T / np.sqrt(D)
                if causal:
                    s[np.arange(Skv)[None, :] > np.arange(Sq)[:, None] + Skv - Sq] = -np.inf
                p = np.exp(s - s.max(axis=1, keepdims=True))
                out[b, :, h] = p @ v[b, :, h // group].astype(np.float64) / p.sum(axis=1, keepdims=True)
    return out


def _inputs(seed, B, Sq, Skv, Hq, Hkv, D):
    return (prng.normal(seed, (B, Sq, Hq, D)), prng.normal(seed + 1, (B, Skv, Hkv, D)),
            prng.normal(seed + 2, (B, Skv, Hkv, D)))


# (B, Sq, Skv, Hq, Hkv): D = 64 takes this kernel from 257 tiles of 64 queries
SHAPES = [
    (1, 129, 129, 3, 3),     # a second tile of one query
    (1, 33, 65, 4, 2),       # a third key block of one key
    (2, 127, 190, 4, 1),     # the last key block two short, a group of four
    (1, 1, 513, 2, 2),       # one query
    (9, 130, 130, 16, 8),    # more than 256 tiles: one group of waves
    (5, 200, 223, 32, 8),
]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_attention_split_shapes(dev, shape, D, causal):
    case(f"attention split {shape} D={D} causal={causal}")
    q, k, v = _inputs(4000 + D, *shape, D)
    got = _run(dev, q, k, v, causal)
    assert oracle.normwise_error(got, _ref(q, k, v, causal)) <= oracle.tolerance(max(shape[2], D))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_attention_split_non_finite(dev, D, causal):
    """Infinite and NaN inputs and values above the largest bf16 reach the
    rows and columns that fp32 arithmetic takes them to, and no others: a key
    that scores minus infinity has probability 0, one that scores plus
    infinity or NaN spoils the row."""
    B, Sq, Skv, Hq, Hkv = 9, 130, 150, 16, 16
    case(f"attention split non-finite D={D} causal={causal}")
    q, k, v = _inputs(5000 + D, B, Sq, Skv, Hq, Hkv, D)
    k[0, 3, 1, 5] = -np.inf
    q[1, 7, 2, 0] = np.nan
    v[2, 9, 3, 4] = np.inf
    v[3, 11, 4, 6] = np.float32(3.4e38)  # rounds to infinity as bf16
    got, ref = _run(dev, q, k, v, causal), _ref(q, k, v, causal)
    # (probability 0 times an infinite value is NaN where the kernel reaches
    # the key: the fp64 sums decide it the same way for unmasked keys only)
    skip = np.zeros(got.shape, bool)
    if causal:
        skip[2, :, 3, 4] = True
    finite = np.isfinite(ref) & ~skip
    assert np.array_equal(np.isnan(got) & ~skip, np.isnan(ref) & ~skip)
    inf = np.isinf(ref) & ~skip
    assert np.array_equal(got[inf], ref[inf].astype(np.float32))
    big = np.zeros(got.shape, bool)
    big[3, :, 4, 6] = True
    for part in (finite & ~big, finite & big):
        scale = 2.0 ** -100 if (part & big).any() else 1.0
        err = oracle.normwise_error(np.where(part, got, 0.0).astype(np.float64) * scale, np.where(part, ref, 0.0) * scale)
        assert err <= oracle.tolerance(Skv)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("q_exp,k_exp,v_exp", [(0, 0, 0), (0, 0, -118), (0, 0, 100), (-118, 118, 0), (118, -118, 0), (90, -90, -100)])
def test_attention_split_range(dev, q_exp, k_exp, v_exp, D, causal):
    """Operands at the ends of fp32's range whose scores are ordinary: each
    keeps its 24 bits.  A score rounds as a sum over D, and its probability by
    that times its size (at most 4 or so)."""
    shape = (9, 130, 150, 16, 16)
    case(f"attention split range D={D} causal={causal} 2^{q_exp} 2^{k_exp} 2^{v_exp}")
    q, k, v = _inputs(4100 + D, *shape, D)
    two = np.float32(2.0)
    q, k, v = q * two ** np.float32(q_exp), k * two ** np.float32(k_exp), v * two ** np.float32(v_exp)
    got = _run(dev, q, k, v, causal)
    assert "attention_split" in _run.kernel, _run.kernel
    assert two_norm_error(got, _ref(q, k, v, causal)) <= fp32_sum_error(shape[2]) + 4 * fp32_sum_error(D)


@pytest.mark.parametrize("block", [4, 5])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_attention_split_non_finite_two_groups(dev, D, causal, block):
    """One group of waves (even or odd key blocks) recomputes in fp32 and
    hands over to, or takes from, the group that did not."""
    B, S, H = 1, 1100, 16
    case(f"attention split non-finite, two groups, D={D} causal={causal} block {block}")
    q, k, v = _inputs(5100 + D, B, S, S, H, H, D)
    key = 32 * block + 5
    v[0, key, 3, 4] = np.float32(3.4e38)       # finite everywhere, beyond the scaled range
    v[0, key, 5, 6] = np.inf
    k[0, key, 7, 8] = np.float32(2.0 ** 113)   # scores of +-2^113 or so: the key takes all or nothing
    got, ref = _run(dev, q, k, v, causal), _ref(q, k, v, causal)
    assert _run.kernel == f"attention_split D={D} x2"
    if causal:  # (probability 0 times infinity is NaN where the kernel reaches a masked key)
        got[0, :key, 5, 6] = ref[0, :key, 5, 6] = 0.0
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert inf.any() and np.array_equal(got[inf], ref[inf].astype(np.float32))
    big = np.isfinite(ref) & (np.abs(ref) > 1e20)
    assert big.any()
    for part, scale in ((big, 2.0 ** -100), (np.isfinite(ref) & ~big, 1.0)):
        err = two_norm_error(got[part].astype(np.float64) * scale, ref[part] * scale)
        assert err <= fp32_sum_error(S) + 4 * fp32_sum_error(D)
