"""The flat parallel-beam kernels (rays within slices of constant z) on the GPU.

Every form that they accept is compared with the FP64 oracle and with the
general kernels in FP64 (the FP32 ones for general geometries place samples
of a 257-slice volume up to 7e-6 of the norm off themselves). Tolerance: FP32 positions are off by at most N / 2^24 voxel
(N <= 160 here: 1e-5), which moves a sample of unit-variance data by about as
much, and the errors of the N samples of a ray or of the angles of a voxel
average out as 1 / sqrt(N); the FP32 sums add sqrt(N) / 2^24. Both stay below
2e-6 of the result's norm.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2
from tomosipo_amd.torch_support import to_autograd

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = 2e-6


def _scan(shape, det, angles, pitch=1.0, pitch_v=None, voxel=(1.0, 1.0, 1.0), flip=(1, 1), skew=0.0, order=None,
          turn=np.pi):
    """A flat parallel scan: `angles` directions over `turn` (in the order `order`), pixels of `pitch`
    voxels, u leaving the slices by `skew` of its length."""
    n = angles if np.isscalar(angles) else len(angles)
    theta = (np.arange(n) + 0.3) * turn / n if np.isscalar(angles) else np.asarray(angles, dtype=float)
    if order is not None:
        theta = theta[np.random.default_rng(order).permutation(n)]
    zero = np.zeros(n)
    pv = pitch if pitch_v is None else pitch_v
    ray = np.stack([zero, np.cos(theta), np.sin(theta)], 1)
    u = flip[1] * pitch * np.stack([zero + skew, -np.sin(theta), np.cos(theta)], 1)
    v = flip[0] * pv * np.stack([zero + 1, zero, zero], 1)
    pos = np.stack([zero + 0.13, 0.2 * np.sin(3 * theta), 0.1 * np.cos(theta)], 1)  # (an uneven mount)
    vg = ts.volume(shape=shape, size=tuple(s * w for s, w in zip(shape, voxel)))
    return vg, ts.parallel_vec(shape=det, ray_dir=ray, det_pos=pos, det_v=v, det_u=u)


CASES = {
    "cube": dict(shape=(64, 64, 64), det=(64, 96), angles=24),
    "one_slice": dict(shape=(1, 40, 44), det=(1, 61), angles=33),
    "ragged": dict(shape=(75, 41, 53), det=(77, 61), angles=19),
    "two_per_lane": dict(shape=(65, 20, 18), det=(66, 25), angles=10),
    "four_per_lane": dict(shape=(129, 20, 24), det=(131, 33), angles=11),
    "two_chunks": dict(shape=(257, 12, 16), det=(250, 19), angles=9),
    "fine_columns": dict(shape=(20, 33, 31), det=(21, 67), angles=21, pitch=0.6, pitch_v=1.0),
    "fine_both": dict(shape=(70, 33, 31), det=(99, 51), angles=21, pitch=0.8),
    "finer_than_half": dict(shape=(20, 17, 19), det=(21, 71), angles=12, pitch=0.37, pitch_v=1.0),
    "coarse": dict(shape=(70, 48, 48), det=(31, 25), angles=24, pitch=2.4),
    "coarser": dict(shape=(20, 64, 64), det=(21, 15), angles=24, pitch=6.0, pitch_v=1.0),
    "fine_rows": dict(shape=(70, 20, 20), det=(300, 30), angles=8, pitch_v=0.24),
    "few_angles": dict(shape=(70, 64, 64), det=(70, 96), angles=3),
    "one_angle": dict(shape=(70, 24, 24), det=(70, 36), angles=[0.4]),
    "one_axis": dict(shape=(70, 24, 24), det=(70, 36), angles=np.linspace(-0.7, 0.7, 12)),
    "along_axes": dict(shape=(70, 24, 28), det=(70, 36), angles=[0.0, np.pi / 2, np.pi, 1.5 * np.pi]),
    "shuffled": dict(shape=(70, 40, 40), det=(70, 60), angles=40, order=3, turn=2 * np.pi),
    "flipped": dict(shape=(70, 24, 24), det=(60, 36), angles=13, flip=(-1, -1)),
    "skewed": dict(shape=(66, 24, 24), det=(70, 36), angles=13, skew=0.2),
    "voxels": dict(shape=(66, 24, 30), det=(70, 45), angles=13, voxel=(0.7, 1.2, 0.9), pitch=1.1),
    "narrow": dict(shape=(70, 48, 48), det=(20, 7), angles=17),
    "three_slices": dict(shape=(3, 40, 44), det=(3, 131), angles=33),
    "eight_slices": dict(shape=(8, 70, 66), det=(9, 300), angles=66),
    "longest_chunk": dict(shape=(127, 20, 24), det=(131, 33), angles=11),
    "aligned_chunks": dict(shape=(192, 20, 24), det=(180, 150), angles=35),
    "many_angles": dict(shape=(4, 16, 16), det=(4, 24), angles=300),
    "many_angles_long": dict(shape=(150, 8, 8), det=(150, 40), angles=170),
}


@pytest.mark.parametrize("case", list(CASES))
def test_flat_kernels_match_oracle_and_general_kernels(case):
    vg, pg = _scan(**CASES[case])
    A = ts.operator(vg, pg)
    g = oracle.oracle_geometry(vg, pg)
    rng = np.random.default_rng(5)
    x = rng.standard_normal(A.domain_shape).astype(np.float32)
    y = rng.standard_normal(A.range_shape).astype(np.float32)
    xd, yd = torch.from_numpy(x).to(DEV), torch.from_numpy(y).to(DEV)
    f, b = A(xd), A.T(yd)
    e = rel_l2(f.cpu().numpy(), oracle.fp(g, x)), rel_l2(b.cpu().numpy(), oracle.bp(g, y))
    f0, b0 = to_autograd(A, dtype=torch.float64)(xd.double()), to_autograd(A.T, dtype=torch.float64)(yd.double())
    d = rel_l2(f.cpu().numpy(), f0.cpu().numpy()), rel_l2(b.cpu().numpy(), b0.cpu().numpy())
    print(f"[flat] {case}: fp {e[0]:.1e}, bp {e[1]:.1e} (oracle), {d[0]:.1e}, {d[1]:.1e} (general kernels)", flush=True)
    assert max(e) <= TOL and max(d) <= 2 * TOL


@pytest.mark.parametrize("shape,det,batch", [((1, 20, 24), (1, 30), 17), ((1, 20, 20), (1, 30), 65),
                                             ((13, 20, 20), (12, 30), 5), ((33, 16, 20), (33, 30), 9)])
def test_flat_batches_equal_single_calls(shape, det, batch):
    """Batch entries share the lines (short ones pass from the kernels without staging to those
    with it): every entry equals its own call bitwise, plain and with each epilogue."""
    from tomosipo_amd.fused import Epilogue, fused_backward, fused_forward

    A = ts.operator(*_scan(shape, det, 15))
    plan = A.projector.plan(0)
    s = torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=DEV)
    gen.manual_seed(batch)
    xs = torch.randn((batch,) + A.domain_shape, generator=gen, device=DEV)
    ys = torch.randn((batch,) + A.range_shape, generator=gen, device=DEV)
    fs, bs = torch.empty_like(ys), torch.empty_like(xs)
    plan.forward(xs.data_ptr(), fs.data_ptr(), False, s, batch, xs[0].numel(), ys[0].numel())
    plan.backward(bs.data_ptr(), ys.data_ptr(), False, s, batch, xs[0].numel(), ys[0].numel())
    f1, b1 = fused_forward([A] * batch, list(xs)), fused_backward([A] * batch, list(ys))
    for k in range(batch):
        f, b = A(xs[k]), A.T(ys[k])
        assert torch.equal(fs[k], f) and torch.equal(bs[k], b), k
        assert torch.equal(f1[k], f) and torch.equal(b1[k], b), k
    # epilogues: the same sums, written as asked
    w, c = torch.rand_like(ys[0]), torch.rand_like(xs[0])
    f, b = A(xs[0]), A.T(ys[0])
    out = fused_forward([A] * 2, [xs[0]] * 2, out=[ys[1].clone(), torch.empty_like(w)],
                        epilogues=[Epilogue("add"), Epilogue("residual", y=ys[0], w=w)])
    assert torch.equal(out[0], ys[1] + f) and rel_l2(out[1].cpu().numpy(), (w * (ys[0] - f)).cpu().numpy()) <= 1e-6
    out = fused_backward([A] * 2, [ys[0]] * 2, out=[xs[1].clone(), xs[1].clone()],
                         epilogues=[Epilogue("add"), Epilogue("scaled_add", w=c)])
    assert torch.equal(out[0], xs[1] + b) and rel_l2(out[1].cpu().numpy(), (xs[1] + c * b).cpu().numpy()) <= 1e-6


@pytest.mark.parametrize("shape,det", [((20, 24, 24), (20, 36)), ((70, 24, 24), (70, 36))])
def test_infinite_pixels_reach_only_their_rays_voxels(shape, det):
    A = ts.operator(*_scan(shape, det, 12, pitch=1.3))
    y = torch.zeros(A.range_shape, device=DEV)
    y[det[0] // 2, 5, det[1] // 2] = 1.0
    met = A.T(y) > 0
    y[det[0] // 2, 5, det[1] // 2] = float("inf")
    b = A.T(y)
    assert met.any() and torch.equal(~torch.isfinite(b), met)
    x = torch.ones(A.domain_shape, device=DEV)
    x[3, 4, 5] = float("nan")
    seen = torch.zeros_like(x)
    seen[3:4, 4:5, 5:6] = 1.0
    hit = A(seen) != 0
    assert torch.isfinite(A(x)).any() and torch.isnan(A(x))[hit].all()
