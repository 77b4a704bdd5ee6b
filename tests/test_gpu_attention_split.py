"""The split-product attention kernel (lancius_amd/csrc/attention_split.hip):
ragged query and key counts at the edges of its tiles, each head dim, both
grids (one tile per CU, and more), and non-finite inputs, against fp64."""
import numpy as np
import pytest
import torch

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


# grids of at most 256 tiles whatever D (D = 64: more than 256 of 64 queries):
# two groups of waves take the even and the odd key blocks
TWO_GROUPS = [
    (1, 1100, 1100, 16, 16),  # an even number of key blocks less four keys
    (1, 1089, 1121, 16, 4),   # an odd number and one key, a last tile of 65 queries
    (2, 640, 1000, 16, 8),
]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("shape", TWO_GROUPS, ids=["x".join(map(str, s)) for s in TWO_GROUPS])
def test_attention_split_two_groups(dev, shape, D, causal):
    case(f"attention split, two groups, {shape} D={D} causal={causal}")
    q, k, v = _inputs(4200 + D, *shape, D)
    got = _run(dev, q, k, v, causal)
    assert _run.kernel == f"attention_split D={D} x2"
    assert two_norm_error(got, _ref(q, k, v, causal)) <= fp32_sum_error(shape[2]) + 4 * fp32_sum_error(D)


def _low(rng_seed, n):
    """n numbers and their first two bf16 parts."""
    x = torch.from_numpy(prng.normal(rng_seed, (n,)))
    h = x.bfloat16().float()
    return tuple(t.numpy() for t in (x, h, (x - h).bfloat16().float()))


@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_attention_split_scores_keep_their_low_products(dev, D):
    """Scores whose four terms x y - h yh - h ym - m yh (h, m: the first two
    bf16 parts) leave what the parts' last products add, about 2^-16, scaled
    up to ordinary size: without one of hl', mm', lh' a score is off by as much
    as it is; with them by the fp32 sum's rounding, 2^-24 of xy, 2^-8 of it."""
    B, S, H = 9, 150, 16
    case(f"attention split low products of the scores D={D}")
    n = B * S * H
    x, xh, xm = _low(4301, n * D // 4)
    y, yh, ym = _low(4302, n * D // 4)
    q = np.stack([x, -xh, -xh, -xm], -1).reshape(B, S, H, D)
    k = np.stack([y, yh, ym, yh], -1).reshape(B, S, H, D)
    # one key row per head serves every query: the terms have to belong together
    k[:] = k[:, :1]
    q64 = q.reshape(B, S, H, D // 4, 4).astype(np.float64)
    y64 = k.reshape(B, S, H, D // 4, 4)[:, :1].astype(np.float64)
    assert np.abs((q64 * y64).sum(-1)).max() < 2.0 ** -11
    # half of the keys are zero: their score is 0, the others' what is left
    k[:, ::2] = 0.0
    v = prng.normal(4303, (B, S, H, D))
    scale = 2.0 ** 16 / np.sqrt(D)
    dq, dk, dv, do = dev.upload(q), dev.upload(k), dev.upload(v), dev.alloc(q.nbytes)
    dev.attention_gqa(do, dq, dk, dv, B, S, S, H, H, D, False, scale)
    assert "attention_split" in dev.launched()[0]
    got = dev.download(do, q.shape)
    for b in (dq, dk, dv, do):
        b.free()
    ref = _ref(q * np.float64(scale * np.sqrt(D)), k, v, False)
    assert two_norm_error(got, ref) <= 2.0 ** -6


@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_attention_split_keeps_constant_values(dev, D):
    """The weighted mean of one value is that value: probabilities lose no more
    than their own rounding on the way into the products, and V nothing (a row
    that sees one key is V bit for bit)."""
    B, S, H = 9, 150, 16
    case(f"attention split constant values D={D}")
    q, k, v = _inputs(4400 + D, B, S, S, H, H, D)
    v[:] = v[:, :1]
    got = _run(dev, q, k, v, True)
    assert "attention_split" in _run.kernel
    assert np.array_equal(got[:, 0], v[:, 0])
    # Rows of up to eight keys: numerator, sum, reciprocal and product round by
    # at most 2^-24 each, the numerator's matrix sum up to three times (1.0 rms
    # and 4.1 at most measured, in 2^-24); a probability short of its third part
    # is off by 2^-18 or so, 38 rms of one key.  Later rows round once more a step.
    err = 2.0 ** 24 * np.abs(got.astype(np.float64) - v) / np.abs(v)
    assert err[:, 1:8].max() <= 6 and np.sqrt(np.mean(err[:, 1:8] ** 2)) <= 2
    assert err.max() <= 6 + 2 * S / 32


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
