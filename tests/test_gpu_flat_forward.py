"""Forms of the flat forward projector on the GPU.

One, two and four values per lane; a lane or several per ray; four angles or one per
block; one layout of the volume or one for either stepping axis; offsets beyond 24
bits. Against the FP64 oracle with the tolerance of the flat kernels' own tests
(2e-6 of the result's norm), and batches bitwise against single calls, which
take other forms.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operator(shape, det, theta, pitch=1.0, pitch_v=None):
    n = max(shape[1:])
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    pv = pitch if pitch_v is None else pitch_v
    pg = ts.parallel(angles=theta, shape=det, size=(pv * det[0] / n, pitch * det[1] / n))
    return ts.operator(vg, pg)


def _around(angles):
    return (np.arange(angles) + 0.3) * np.pi / angles


CASES = {
    # (blocks of four angles: 64 columns of them are one tile of a single slice)
    "one_w_four_angles": ((1, 16, 18), (1, 600), _around(1800)),
    "two_w_four_angles": ((2, 16, 18), (2, 600), _around(1800)),
    "four_w_four_angles": ((4, 16, 18), (4, 600), _around(700)),
    "rays_of_lanes_four_angles": ((15, 16, 18), (15, 300), _around(500)),
    "sixteen_w_four_angles": ((16, 16, 18), (16, 300), _around(400)),
    "one_w_one_axis": ((1, 40, 37), (1, 70), np.linspace(-0.7, 0.7, 9)),
    "two_w_other_axis": ((2, 40, 37), (2, 70), np.pi / 2 + np.linspace(-0.7, 0.7, 9)),
    "three_w": ((3, 70, 33), (3, 70), _around(21)),
    "five_w": ((5, 33, 70), (5, 71), _around(21)),
    "many_groups": ((1, 300, 20), (1, 330), _around(17)),
    "groups_for_four_waves": ((2, 129, 257), (2, 300), _around(13)),
    "narrow_detector": ((1, 50, 50), (1, 3), _around(30)),
    "wide_detector": ((1, 8, 8), (1, 200), _around(30)),
}


@pytest.mark.parametrize("case", list(CASES))
def test_forward_forms_match_oracle(case):
    A = _operator(*CASES[case])
    x = np.random.default_rng(8).standard_normal(A.domain_shape).astype(np.float32)
    y = A(torch.from_numpy(x).to(DEV)).cpu().numpy()
    e = rel_l2(y, oracle.fp(oracle.oracle_geometry(A.volume_geometry, A.projection_geometry), x))
    print(f"[flat forward] {case}: {e:.1e}", flush=True)
    assert e <= 2e-6


def test_forward_offsets_beyond_24_bits():
    """Neighbouring voxel columns of y-stepping rays lie 1024 lines of 4100 floats apart (17 MB)."""
    A = _operator((4100, 1024, 2), (5, 6), np.pi / 2 + np.array([-0.4, -0.001, 0.002, 0.5]), 0.7, 800.0)
    x = np.random.default_rng(8).standard_normal(A.domain_shape).astype(np.float32)
    y = A(torch.from_numpy(x).to(DEV)).cpu().numpy()
    assert rel_l2(y, oracle.fp(oracle.oracle_geometry(A.volume_geometry, A.projection_geometry), x)) <= 2e-6


@pytest.mark.parametrize("shape,det,batches", [((1, 70, 65), (1, 90), (2, 3, 4, 5, 15, 16, 31, 65, 130)),
                                               ((2, 30, 33), (3, 40), (2, 7, 8, 40)), ((7, 40, 30), (6, 50), (2, 3, 20))])
def test_batches_hold_the_bits_of_single_calls(shape, det, batches):
    from tomosipo_amd.fused import fused_forward

    A = _operator(shape, det, _around(23))
    plan, s = A.projector.plan(0), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=DEV)
    gen.manual_seed(shape[1])
    xs = torch.randn((max(batches),) + A.domain_shape, generator=gen, device=DEV)
    want = [A(xs[k]) for k in range(max(batches))]
    for batch in batches:
        out = torch.empty((batch,) + A.range_shape, device=DEV)
        plan.forward(xs.data_ptr(), out.data_ptr(), False, s, batch, xs[0].numel(), out[0].numel())
        for k in range(batch):
            assert torch.equal(out[k], want[k]), (batch, k)
        fused = fused_forward([A] * batch, list(xs[:batch]))
        assert all(torch.equal(f, w) for f, w in zip(fused, want)), batch


def test_non_finite_voxels_reach_their_rays_only():
    """A NaN voxel: exactly the rays with a weight on it, found with the voxel set to one; for one, two
    and more values per lane."""
    for nz in (1, 2, 5, 20, 70):
        A = _operator((nz, 24, 21), (nz, 36), _around(12), 1.3)
        seen = torch.zeros(A.domain_shape, device=DEV)
        seen[nz // 2, 5, 6] = 1.0
        hit = A(seen) != 0
        x = torch.ones(A.domain_shape, device=DEV)
        x[nz // 2, 5, 6] = float("nan")
        nan = torch.isnan(A(x))
        # (a ray through the exact edge of the voxel's tent has weight 0 and may read it)
        assert hit.any() and nan[hit].all() and int((nan & ~hit).sum()) <= int(hit.sum()) // 10 + 2
        assert not nan.all()
