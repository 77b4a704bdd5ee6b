"""Column sums (lancius_amd/csrc/reduce.hip) and the cross-entropy loss
(rowops.hip) where their forms change, against fp64."""
import numpy as np
import pytest

from lancius_amd import prng
from tests.conftest import case

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (7, 16), (8, 17), (31, 15), (63, 33), (65, 64), (511, 65), (512, 300), (513, 5), (2048, 16), (2049, 16),
          (1025, 32), (4100, 130), (48, 65536), (49, 65536), (48, 65535), (3, 70001), (9000, 1000)]


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_sum_axis0_forms(dev, rows, cols):
    case(f"sum_axis0 {rows}x{cols}")
    x = prng.normal(9000, (rows, cols))
    dx, do = dev.upload(x), dev.alloc(4 * cols + 256)
    dev.fill(do, 7.0, cols + 64)
    dev.sum_axis0(do, dx, rows, cols)
    got = dev.download(do, (cols + 64,))
    dx.free(), do.free()
    assert (got[cols:] == 7.0).all()
    exact = x.astype(np.float64).sum(0)
    # summed in fp64 and rounded once: half an ulp, and the fp64 sums' own error
    bound = np.abs(exact) * 2.0**-24 + np.abs(x).sum(0, dtype=np.float64) * rows * 2.0**-53
    assert (np.abs(got[:cols] - exact) <= bound).all()


@pytest.mark.parametrize("rows", [1, 15, 33, 64, 65, 256, 257, 8193])
@pytest.mark.parametrize("cols", [1, 16, 17, 64, 65, 256, 257])
def test_cross_entropy_forms(dev, rows, cols):
    case(f"cross_entropy {rows}x{cols}")
    x = prng.normal(9100, (rows, cols), std=3.0)
    y = np.zeros((rows, cols), np.float32)
    y[np.arange(rows), (np.arange(rows) * 7) % cols] = 1.0
    y[0] = 0.0  # a row without a target adds nothing
    dx, dy, do = dev.upload(x), dev.upload(y), dev.alloc(4)
    dev.cross_entropy(do, dx, dy, rows, cols)
    got = float(dev.download(do, (1,))[0])
    for b in (dx, dy, do):
        b.free()
    x64 = x.astype(np.float64)
    m = x64.max(1)
    lse = m + np.log(np.exp(x64 - m[:, None]).sum(1))
    want = abs(((x64 - lse[:, None]) * y).sum() / rows)
    # per row: the fp32 sum of exponentials (cols + 4 roundings), its logarithm, an ulp of the result
    assert abs(got - want) <= (cols + 8) * 2.0**-23 + abs(want) * 2.0**-23
