"""The upright FDK backprojector on the GPU against the FP64 oracle.

Pixels of about a voxel (32 voxels per column), fine ones (8), and so fine ones
that an angle's pixels do not fit LDS; a source between the volume's corners
(voxels behind it); volumes that are no multiple of a block; detectors that the
shadow leaves on every side. Tolerance: rows relative to a block's first are
FP32 below 62, 4e-6 of a pixel with their steps, on independent random
pixels: below 1e-5 of the result's norm.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from oracle import fdk as F
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape, det, size, distance", [
    ((33, 17, 35), (48, 60), (1.4, 1.8), 2.5), ((7, 16, 16), (9, 40), (1.2, 1.6), 2.5),
    ((65, 32, 31), (20, 24), (0.6, 0.7), 2.5), ((40, 40, 40), (130, 150), (1.3, 1.7), 2.5),
    ((40, 40, 40), (500, 600), (1.3, 1.7), 2.5), ((64, 20, 24), (70, 60), (1.3, 1.7), 0.62),
    ((24, 20, 24), (30, 60), (1.3, 1.7), 0.4)])
def test_upright_backprojection_matches_oracle(shape, det, size, distance, monkeypatch):
    n = max(shape)
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    pg = ts.cone(angles=9, shape=det, size=size, src_orig_dist=distance, src_det_dist=distance)
    A = ts.operator(vg, pg)
    y = np.random.default_rng(2).random(A.range_shape, dtype=np.float32)
    out = ts.fdk(A, torch.from_numpy(y).cuda())
    if distance < 0.5:
        # (the oracle also counts voxels behind the source, which both kernels leave out)
        monkeypatch.setenv("TSX_FORCE_GENERAL", "1")
        ref = ts.fdk(A, torch.from_numpy(y).cuda()).cpu().numpy()
    else:
        ref = F.fdk(oracle.oracle_geometry(vg, pg), y)
    assert rel_l2(out.cpu().numpy(), ref) <= 1e-5
