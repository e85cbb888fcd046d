"""Parallel scans cut into z-slabs, angle ranges and batches (GPU).

On the padded and the separable kernels, which these scans run where a variable
asks for them, and on the flat ones: angle ranges of the backprojector, and
batches cut where a launch's turned volume would pass 4 GiB. Tolerances as in
the other chunked tests: 1e-5 against the oracle, 1e-6 between chunked and
unchunked sums of one kernel.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"
LIMIT = 400000


@pytest.mark.parametrize("flat", [False, True])
def test_slabs_and_angle_ranges_of_a_parallel_scan(monkeypatch, flat):
    vg = ts.volume(shape=48, size=1)
    pg = ts.parallel(angles=40, shape=(48, 72), size=(1, 1.5))
    monkeypatch.setenv("TSX_CHUNK_BYTES", str(LIMIT))
    A = ts.operator(vg, pg)
    A.projector.plan(0)
    monkeypatch.delenv("TSX_CHUNK_BYTES")
    B = ts.operator(vg, pg)
    if not flat:
        monkeypatch.setenv("TSX_FP_VARIANT", "4")
        monkeypatch.setenv("TSX_BP_BRICK_Z", "32")
    info = A.projector.plan(0).info()
    assert (info["fp_flat"], info["bp_flat"]) == (flat, flat)
    assert info["fp_slabs"] == 3 and info["bp_launch_angles"] == 25
    rng = np.random.default_rng(12)
    x = rng.random(A.domain_shape).astype(np.float32)
    y = rng.random(A.range_shape).astype(np.float32)
    xd, yd = torch.from_numpy(x).to(DEV), torch.from_numpy(y).to(DEV)
    g = oracle.oracle_geometry(vg, pg)
    f, b = A(xd).cpu().numpy(), A.T(yd).cpu().numpy()
    assert rel_l2(f, oracle.fp(g, x)) <= 1e-5 and rel_l2(b, oracle.bp(g, y)) <= 1e-5
    assert rel_l2(f, B(xd).cpu().numpy()) <= 1e-6 and rel_l2(b, B.T(yd).cpu().numpy()) <= 1e-6


def test_batches_whose_turned_volume_passes_4_gib():
    """Two slices of 5792^2, 17 entries: 4.6 GB of turned volume, cut into launches of 15 or 16 entries and the
    rest. Entries hold two different volumes in turn, compared with their single calls bitwise."""
    n, angles, batch = 5792, 3, 17
    vg = ts.volume(shape=(2, n, n), size=(2 / n, 1, 1))
    A = ts.operator(vg, ts.parallel(angles=np.array([0.3, 1.1, 2.0]), shape=(2, 700), size=(2 / n, 1.4)))
    plan, s = A.projector.plan(0), torch.cuda.current_stream().cuda_stream
    assert plan.info()["fp_flat"]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(3)
    pair = torch.rand((2,) + A.domain_shape, generator=gen, device=DEV)
    want = [A(pair[0]), A(pair[1])]
    xs = pair.repeat((batch + 1) // 2, 1, 1, 1)[:batch].contiguous()
    out = torch.empty((batch,) + A.range_shape, device=DEV)
    plan.forward(xs.data_ptr(), out.data_ptr(), False, s, batch, xs[0].numel(), out[0].numel())
    for k in range(batch):
        assert torch.equal(out[k], want[k % 2]), k


def test_more_instances_than_a_launch_holds():
    """37 flat scans of different sizes, each way: three launches of at most sixteen, angle parts among them."""
    from tomosipo_amd.fused import fused_backward, fused_forward

    ops = []
    for k in range(37):
        shape = ((3, 20, 70, 33)[k % 4], 20 + k, 18 + 2 * (k % 5))
        vg = ts.volume(shape=shape, size=tuple(v / 40 for v in shape))
        ops.append(ts.operator(vg, ts.parallel(angles=12 + k, shape=(shape[0] + k % 3, 50), size=(shape[0] / 40, 1.4))))
    gen = torch.Generator(device=DEV)
    gen.manual_seed(9)
    xs = [torch.randn(A.domain_shape, generator=gen, device=DEV) for A in ops]
    ys = [torch.randn(A.range_shape, generator=gen, device=DEV) for A in ops]
    assert all(A.projector.plan(0).info()["fp_flat"] for A in ops)
    for A, x, got in zip(ops, xs, fused_forward(ops, xs)):
        assert torch.equal(got, A(x))
    for A, y, got in zip(ops, ys, fused_backward(ops, ys)):
        assert torch.equal(got, A.T(y))
