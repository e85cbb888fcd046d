"""The FDK ramp filter on the GPU (matrix cores) against the FP64 oracle.

Widths on either side of one pass of each tiling (128, 256, 512, 768 columns),
of one column more than the next 16 pixel differences, odd ones and several
passes; row counts on either side of a block's 16. Tolerance: FP32 sums over
the row's pixel differences, 1e-6 relative on rows of independent random
pixels, which the backprojection averages: 2e-6 of the result's norm.
"""
import numpy as np
import pytest

import oracle
import oracle.fdk as F
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _scan(rows, cols, tilt=0.0, angles=5):
    vg = ts.volume(shape=(6, 14, 18), size=(0.4, 0.8, 1))
    pg = ts.cone(angles=angles, shape=(rows, cols), size=(0.6, 1.8), cone_angle=0.3)
    if tilt:
        pg = ts.rotate(pos=0, axis=(0, 1, 0), angles=tilt) * pg.to_vec()
    return vg, pg


@pytest.mark.parametrize("tilt", [0.0, 0.1])
@pytest.mark.parametrize("rows, cols", [(1, 1), (2, 3), (15, 31), (16, 32), (17, 33), (9, 127), (16, 128), (18, 129),
                                        (5, 256), (31, 257), (33, 511), (8, 513), (16, 768), (17, 769), (4, 1601),
                                        (2, 4096)])
def test_filter_matches_oracle(rows, cols, tilt):
    vg, pg = _scan(rows, cols, tilt)
    A = ts.operator(vg, pg)
    y = np.random.default_rng(cols).random(A.range_shape, dtype=np.float32)
    out = ts.fdk(A, torch.from_numpy(y).cuda())
    assert rel_l2(out.cpu().numpy(), F.fdk(oracle.oracle_geometry(vg, pg), y)) <= 2e-6


@pytest.mark.parametrize("cols", [90, 900])
def test_filter_spreads_an_infinite_pixel_as_the_oracle(cols):
    """One infinite pixel: the filtered row is infinite in the columns of the
    other parity, so every voxel that reads that row of that angle is -inf, or
    NaN next to the pixel (which itself is +inf); the others stay finite."""
    vg, pg = _scan(20, cols, angles=3)
    A = ts.operator(vg, pg)
    y = np.random.default_rng(1).random(A.range_shape, dtype=np.float32)
    y[9, 1, cols // 2] = np.inf
    out = ts.fdk(A, torch.from_numpy(y).cuda()).cpu().numpy()
    y[9, 1, cols // 2] = 0.0
    base = ts.fdk(A, torch.from_numpy(y).cuda()).cpu().numpy()
    finite = np.isfinite(out)
    assert finite.any() and np.isneginf(out).any() and not np.isposinf(out).all()
    assert rel_l2(out[finite], base[finite]) <= 2e-6
