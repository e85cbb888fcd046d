"""Tilted parallel scans with directions nearly within the detector's plane, on the GPU.

Those directions put the volume 1e6 to 1e11 pixels beyond the detector, so
that they add nothing; the box of a voxel there has to come out empty. The
result is that of the other directions. Tolerance as for every tilted scan:
2e-6 of the norm on random data.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(20, 24, 32), (95, 96, 97)])
@pytest.mark.parametrize("grazing", [1e-4, 1e-6, 1e-7, 1e-9])
@pytest.mark.parametrize("axis", [1, 2])
def test_grazing_directions_add_nothing(shape, grazing, axis):
    n, rows, cols, angles = max(shape), 40, 56, 7
    theta = (np.arange(angles) + 0.3) * np.pi / angles
    zero, one = np.zeros(angles), np.ones(angles)
    ray = np.stack([zero, np.cos(theta), np.sin(theta)], 1)
    u = 1.3 / n * np.stack([zero, -np.sin(theta), np.cos(theta)], 1)
    v = 1.3 / n * np.stack([one, zero, zero], 1)
    pos = 2.0 * ray  # (the planes lie outside the volume)
    # one direction along the detector's u (or v) but for `grazing`
    ray[3] = n / 1.3 * (u[3] if axis == 1 else v[3]) + grazing * ray[3]
    R = ts.rotate(pos=0, axis=(0, 1, 0), angles=0.3)
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    pg = R * ts.parallel_vec(shape=(rows, cols), ray_dir=ray, det_pos=pos, det_v=v, det_u=u)
    A = ts.operator(vg, pg)
    assert A.projector.plan(0).info()["bp_kernel"] == "general"
    y = np.random.default_rng(3).standard_normal(A.range_shape).astype(np.float32)
    print(f"[far] {shape} {grazing} {axis}", flush=True)
    b = A.T(torch.from_numpy(y).to("cuda")).cpu().numpy()
    assert rel_l2(b, oracle.bp(oracle.oracle_geometry(vg, pg), y)) <= 2e-6
