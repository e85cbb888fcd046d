"""The backprojector of tilted detectors (bp_tilted) on the GPU against the FP64 oracle.

Volumes of the three numbers of voxels per thread (8, 2 and 1) and depths that
are no multiple of them; boxes of two, more and fewer than two pixels; angles
stepping along z; detectors that the volume's shadow leaves; sources next to
the volume. Tolerance: pixel positions are FP64 plus FP32 differences of at
most 8 voxels (1e-6 pixel), weights FP32: below 2e-6 of the result's norm on
random data; 1e-5 with the source a few voxels from the volume, where the
FP32 map from pixels to voxels loses as many digits as it magnifies.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda"


def _scan(beam, shape, det, angles, axis, tilt, pitch, distance=2.8):
    n = max(shape)
    theta = (np.arange(angles) + 0.3) * 2 * np.pi / angles
    zero = np.zeros(angles)
    ray = np.stack([zero, np.cos(theta), np.sin(theta)], 1)
    u = pitch / n * np.stack([zero, -np.sin(theta), np.cos(theta)], 1)
    v = pitch / n * np.stack([zero + 1, zero, zero], 1)
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    if beam == "cone":
        pg = ts.cone_vec(shape=det, src_pos=-distance * ray, det_pos=0 * ray, det_v=v, det_u=u)
    else:
        pg = ts.parallel_vec(shape=det, ray_dir=ray, det_pos=0 * ray, det_v=v, det_u=u)
    return vg, ts.rotate(pos=0, axis=axis, angles=tilt) * pg


CASES = {
    "eight": ("cone", (121, 128, 130), (110, 140), 4, (0, 1, 0), 0.2, 1.5, 2.8, 2e-6),
    "two": ("cone", (95, 96, 97), (90, 100), 6, (0, 1, 0), 0.2, 1.5, 2.8, 2e-6),
    "one": ("cone", (33, 40, 44), (40, 60), 20, (0, 1, 0), 0.3, 1.4, 2.8, 2e-6),
    "eight_parallel": ("parallel", (121, 128, 130), (110, 140), 4, (0, 1, 0), 0.2, 1.5, 0, 2e-6),
    "one_parallel": ("parallel", (33, 40, 44), (40, 60), 20, (0, 1, 1), 0.4, 1.0, 0, 2e-6),
    "rolled": ("cone", (40, 40, 40), (40, 60), 15, (0, 1, 1), 0.6, 1.4, 2.8, 2e-6),
    "fine_pixels": ("cone", (95, 96, 97), (200, 260), 5, (0, 1, 0), 0.2, 0.6, 2.8, 2e-6),
    "coarse_pixels": ("cone", (95, 96, 97), (30, 40), 5, (0, 1, 0), 0.2, 5.0, 2.8, 2e-6),
    "z_stepping": ("cone", (40, 36, 44), (60, 60), 20, (0, 1, 0), 1.2, 1.4, 2.8, 2e-6),
    "z_stepping_parallel": ("parallel", (40, 36, 44), (60, 60), 20, (0, 1, 0), 1.2, 1.4, 0, 2e-6),
    "narrow": ("cone", (95, 96, 97), (20, 12), 6, (0, 1, 0), 0.2, 1.5, 2.8, 2e-6),
    "near_source": ("cone", (40, 40, 40), (40, 60), 15, (0, 1, 0), 0.2, 1.4, 0.85, 1e-5),
}


@pytest.mark.parametrize("case", list(CASES))
def test_tilted_backprojection_matches_oracle(case):
    *scan, tol = CASES[case]
    vg, pg = _scan(*scan)
    A = ts.operator(vg, pg)
    assert A.projector.plan(0).info()["bp_kernel"] == "general"
    y = np.random.default_rng(3).standard_normal(A.range_shape).astype(np.float32)
    yd = torch.from_numpy(y).to(DEV)
    b = A.T(yd)
    e = rel_l2(b.cpu().numpy(), oracle.bp(oracle.oracle_geometry(vg, pg), y))
    print(f"[tilted] {case}: {e:.1e}", flush=True)
    assert e <= tol
    # batch entries and fused instances equal single calls bitwise
    from tomosipo_amd.fused import fused_backward

    ys = torch.stack([yd, 2 * yd, yd - 1])
    out = torch.empty((3,) + A.domain_shape, device=DEV)
    A.projector.plan(0).backward(out.data_ptr(), ys.data_ptr(), False, torch.cuda.current_stream().cuda_stream, batch=3,
                                 vol_stride=b.numel(), proj_stride=yd.numel())
    assert torch.equal(out[0], b) and torch.equal(out[2], A.T(ys[2].contiguous()))
    assert torch.equal(fused_backward([A, A], [yd, ys[1].contiguous()])[0], b)
