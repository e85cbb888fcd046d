"""Tilted backprojections whose voxels meet many detector pixels, on the GPU.

The pixels of a voxel's box are read in groups of four columns: boxes of 3 to
about 14 columns, detectors of few columns and rows (groups that pass their
ends), rows of every length modulo 4. Tolerance as for every tilted scan: 2e-6
of the result's norm on random data.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beam", ["cone", "parallel"])
@pytest.mark.parametrize("shape,det,pitch", [((9, 10, 11), (90, 101), 0.2), ((9, 10, 70), (75, 102), 0.45),
                                             ((12, 12, 12), (40, 43), 0.3), ((11, 12, 9), (24, 28), 0.75),
                                             ((10, 10, 10), (5, 3), 0.4), ((10, 10, 10), (3, 130), 0.15)])
def test_many_pixels_per_voxel(beam, shape, det, pitch):
    n, angles = max(shape), 5
    theta = (np.arange(angles) + 0.3) * 2 * np.pi / angles
    zero, one = np.zeros(angles), np.ones(angles)
    ray = np.stack([zero, np.cos(theta), np.sin(theta)], 1)
    u = pitch / n * np.stack([zero, -np.sin(theta), np.cos(theta)], 1)
    v = pitch / n * np.stack([one, zero, zero], 1)
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    pg = (ts.cone_vec(shape=det, src_pos=-2.8 * ray, det_pos=0 * ray, det_v=v, det_u=u) if beam == "cone"
          else ts.parallel_vec(shape=det, ray_dir=ray, det_pos=0 * ray, det_v=v, det_u=u))
    pg = ts.rotate(pos=0, axis=(0, 1, 0), angles=0.25) * pg
    A = ts.operator(vg, pg)
    assert A.projector.plan(0).info()["bp_kernel"] == "general"
    y = np.random.default_rng(4).standard_normal(A.range_shape).astype(np.float32)
    b = A.T(torch.from_numpy(y).to("cuda")).cpu().numpy()
    assert rel_l2(b, oracle.bp(oracle.oracle_geometry(vg, pg), y)) <= 2e-6
