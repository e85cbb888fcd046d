"""The general backprojector (bp_general) on the GPU against the FP64 oracle.

Volumes of fewer voxels than a block has, of exactly a block's 64 and of odd
numbers beyond it; fewer angles than the block's four groups, one more, and
remainders; batches. Tolerance: the float64 path holds positions, weights and
sums in FP64, with tens of roundings per term and sums of hundreds of terms:
1e-12 of the result's norm.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beam", ["parallel", "cone"])
@pytest.mark.parametrize("shape, angles, ss, batch", [
    ((1, 1, 1), 1, 1, 1), ((4, 4, 4), 3, 1, 2), ((3, 5, 13), 4, 2, 3), ((5, 13, 3), 5, 1, 5), ((7, 11, 31), 11, 1, 1)])
def test_general_backprojection_matches_oracle(beam, shape, angles, ss, batch):
    from tomosipo_amd.torch_support import to_autograd

    n = max(shape)
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    pg = (ts.parallel(angles=angles, shape=(9, 14), size=(1.1, 1.7)) if beam == "parallel"
          else ts.cone(angles=angles, shape=(9, 14), size=(1.1, 1.7), cone_angle=0.4))
    A = ts.operator(vg, pg, detector_supersampling=ss)
    g = oracle.oracle_geometry(vg, pg, ss)
    y = np.random.default_rng(5).random((batch, *A.range_shape))
    b = to_autograd(A.T, num_extra_dims=1, dtype=torch.float64)(torch.from_numpy(y).to("cuda")).cpu().numpy()
    for k in range(batch):
        assert rel_l2(b[k], oracle.bp(g, y[k])) <= 1e-12
