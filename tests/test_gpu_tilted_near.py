"""Tilted backprojections with the source close to the volume's corners, on the GPU.

Their voxels' boxes differ by far, so that each thread takes one voxel; somewhat
farther away several share a set-up again. Tolerance: 1e-5 of the result's norm on
random data, as for every source a few voxels from the volume (the FP32 map from
pixels to voxels loses as many digits as it magnifies), 2e-6 farther away.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,distance,tol", [((95, 96, 97), 0.9, 1e-5), ((41, 128, 130), 0.8, 1e-5),
                                                ((95, 96, 97), 1.6, 2e-6)])
def test_sources_near_the_corners(shape, distance, tol):
    n, angles = max(shape), 5
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    pg = ts.cone(angles=angles, shape=(60, 90), size=(1.4, 2.1), src_orig_dist=distance, src_det_dist=distance)
    A = ts.operator(vg, ts.rotate(pos=0, axis=(0, 1, 0), angles=0.1) * pg.to_vec())
    assert A.projector.plan(0).info()["bp_kernel"] == "general"
    y = np.random.default_rng(5).standard_normal(A.range_shape).astype(np.float32)
    b = A.T(torch.from_numpy(y).to("cuda")).cpu().numpy()
    assert rel_l2(b, oracle.bp(oracle.oracle_geometry(A.volume_geometry, A.projection_geometry), y)) <= tol
