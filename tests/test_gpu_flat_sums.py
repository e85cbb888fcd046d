"""Rounding and outputs of the flat backprojector's angle parts on the GPU.

Against 64 bits its sums may round no more than those of the separable kernel,
which takes the same plans where a brick depth is asked for: 1.05 times its
error, a ratio of two sums over some 1e5 voxels of equally distributed
roundings. Outputs that are not 16-byte aligned, entries farther apart than
their size and volumes of odd sizes are written voxel by voxel and hold the same
bits.
"""
import numpy as np
import pytest

import oracle
import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _operator(shape, det, angles, pitch=1.0):
    n = max(shape[1:])
    vg = ts.volume(shape=shape, size=tuple(s / n for s in shape))
    theta = (np.arange(angles) + 0.3) * np.pi / angles
    return ts.operator(vg, ts.parallel(angles=theta, shape=det, size=(pitch * det[0] / n, pitch * det[1] / n)))


@pytest.mark.parametrize("shape,det,angles", [((128, 128, 128), (128, 192), 180), ((1, 256, 256), (1, 384), 180),
                                              ((61, 173, 160), (60, 230), 66), ((1, 167, 167), (1, 230), 277),
                                              ((64, 64, 64), (64, 96), 96)])
def test_sums_round_no_more_than_the_separable_kernels(monkeypatch, shape, det, angles):
    A = _operator(shape, det, angles)
    y = np.random.default_rng(2).random(A.range_shape).astype(np.float32)
    yd = torch.from_numpy(y).to(DEV)
    want = oracle.bp(oracle.oracle_geometry(A.volume_geometry, A.projection_geometry), y)
    e = rel_l2(A.T(yd).cpu().numpy(), want)
    monkeypatch.setenv("TSX_BP_BRICK_Z", "32")
    e0 = rel_l2(A.T(yd).cpu().numpy(), want)
    print(f"[flat sums] {shape} {angles}: {e:.2e}, separable {e0:.2e}", flush=True)
    assert e <= 1.05 * e0


@pytest.mark.parametrize("shape", [(66, 20, 24), (5, 21, 23), (70, 24, 32)])
def test_outputs_of_any_alignment_and_stride_hold_the_same_bits(shape):
    """nx a multiple of 4 or not, the output 0 to 3 floats past a 16-byte
    boundary, entries 0, 1 or 5 floats farther apart than their size."""
    A = _operator(shape, (shape[0], 36), 40)
    plan, s = A.projector.plan(0), torch.cuda.current_stream().cuda_stream
    n, m = int(np.prod(A.domain_shape)), int(np.prod(A.range_shape))
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1)
    ys = torch.randn((3, m + 5), generator=gen, device=DEV)
    xs = torch.randn((3, n + 5), generator=gen, device=DEV)
    want_b = [A.T(ys[k, :m].reshape(A.range_shape).contiguous()).reshape(-1) for k in range(3)]
    want_f = [A(xs[k, :n].reshape(A.domain_shape).contiguous()).reshape(-1) for k in range(3)]
    for shift in range(4):
        for extra in (0, 1, 5):
            for additive in (False, True):
                out = torch.full((3 * (n + extra) + 8,), 2.0, device=DEV)
                plan.backward(out[shift:].data_ptr(), ys.data_ptr(), additive, s, 3, n + extra, m + 5)
                for k in range(3):
                    got = out[shift + k * (n + extra):][:n]
                    assert torch.equal(got, want_b[k] + 2.0 if additive else want_b[k]), (shift, extra, additive, k)
                assert (out[:shift] == 2.0).all() and (out[shift + 2 * (n + extra) + n:] == 2.0).all()
                out = torch.full((3 * (m + extra) + 8,), 2.0, device=DEV)
                plan.forward(xs.data_ptr(), out[shift:].data_ptr(), additive, s, 3, n + 5, m + extra)
                for k in range(3):
                    got = out[shift + k * (m + extra):][:m]
                    assert torch.equal(got, want_f[k] + 2.0 if additive else want_f[k]), (shift, extra, additive, k)
                assert (out[:shift] == 2.0).all() and (out[shift + 2 * (m + extra) + m:] == 2.0).all()


@pytest.mark.parametrize("nz,n,batches", [(1, 36, (2, 3, 4, 5, 60, 64, 65)), (8, 300, (6, 9)), (3, 30, (2, 21, 22))])
def test_short_and_long_lines_hold_the_same_bits(nz, n, batches):
    """A batch's entries lengthen the lines: through the kernel of short lines, one and four values
    per lane, its angle parts in blocks of their own and in turn, to the one that stages lines."""
    A = _operator((nz, n, n - 3), (nz, n + 9), 50)
    plan, s = A.projector.plan(0), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n)
    ys = torch.randn((max(batches),) + A.range_shape, generator=gen, device=DEV)
    want = [A.T(ys[k]) for k in range(max(batches))]
    for batch in batches:
        out = torch.empty((batch,) + A.domain_shape, device=DEV)
        plan.backward(out.data_ptr(), ys.data_ptr(), False, s, batch, out[0].numel(), ys[0].numel())
        for k in range(batch):
            assert torch.equal(out[k], want[k]), (batch, k)


@pytest.mark.parametrize("nz", [1, 7, 8, 15, 16, 17, 33])
@pytest.mark.parametrize("nx", [1, 15, 17, 30])
def test_rows_of_any_length_hold_the_same_bits(nz, nx):
    """Rows of no multiple of four voxels are written through a tile, 64 lanes' values at a time: lines of
    two and four values per lane, in which a tile holds part of an entry, some, or many."""
    A = _operator((nz, 21, nx), (nz, 34), 24)
    plan, s = A.projector.plan(0), torch.cuda.current_stream().cuda_stream
    n = int(np.prod(A.domain_shape))
    gen = torch.Generator(device=DEV)
    gen.manual_seed(nx)
    most = 530 // nz
    ys = torch.randn((most,) + A.range_shape, generator=gen, device=DEV)
    want = [A.T(ys[k]).reshape(-1) for k in range(most)]
    for batch in (70 // nz + 1, 130 // nz + 1, 270 // nz + 1, most):
        for additive in (False, True):
            out = torch.full((batch * (n + 3) + 8,), 2.0, device=DEV)
            plan.backward(out[1:].data_ptr(), ys.data_ptr(), additive, s, batch, n + 3, ys[0].numel())
            rows = out[1:][:batch * (n + 3)].reshape(batch, n + 3)
            for k in range(batch):
                assert torch.equal(rows[k, :n], want[k] + 2.0 if additive else want[k]), (batch, additive, k)
            assert (out[0] == 2.0) and (rows[:, n:] == 2.0).all()


@pytest.mark.parametrize("nz", [1, 2, 3, 4, 7, 20, 24, 36, 41, 48, 61, 64])
@pytest.mark.parametrize("pitch,pixels", [(1.3, 40), (0.8, 60), (0.55, 90)])
def test_short_lines_match_oracle(nz, pitch, pixels):
    """Lines of 1 to 64 (lanes per voxel column from 1 to 16, tiles of every width), two to four detector
    columns per voxel. Tolerance: that of the flat kernels' own tests, 2e-6 of the result's norm."""
    A = _operator((nz, 33, 29), (nz + 1, pixels), 21, pitch)
    y = np.random.default_rng(nz).standard_normal(A.range_shape).astype(np.float32)
    b = A.T(torch.from_numpy(y).to(DEV)).cpu().numpy()
    assert rel_l2(b, oracle.bp(oracle.oracle_geometry(A.volume_geometry, A.projection_geometry), y)) <= 2e-6


@pytest.mark.parametrize("nz", [1, 5, 30])
def test_infinite_pixels_in_short_lines(nz):
    A = _operator((nz, 24, 24), (nz, 36), 12, 1.3)
    y = torch.zeros(A.range_shape, device=DEV)
    y[nz // 2, 5, 18] = 1.0
    met = A.T(y) > 0
    y[nz // 2, 5, 18] = float("inf")
    b = A.T(y)
    assert met.any() and torch.equal(~torch.isfinite(b), met)
