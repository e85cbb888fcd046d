"""tsx_direct_fpbp3d_noalloc on parallel scans whose flat kernels want more scratch than its buffer holds (GPU).

Their forward projections take the angles in more launches; plans whose
backprojection lines do not fit keep the separable kernel, also where another
plan (refined detector, swapped axes) puts its own bytes first. Results are
bitwise those of tsx_direct_fpbp3d, and everything that fits the buffer with the
padded and separable kernels is accepted.
"""
import ctypes

import numpy as np
import pytest

import tomosipo_amd as ts
from tests.conftest import rel_l2
from tomosipo_amd import _tsx

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"
FP, BP = _tsx.TSX_OP_FP, _tsx.TSX_OP_BP


def _scan(shape, det, angles, turned=False):
    vg = ts.volume(shape=shape, size=tuple(s / max(shape) for s in shape))
    pg = ts.parallel(angles=(np.arange(angles) + 0.3) * np.pi / angles, shape=det,
                     size=(1.0, det[1] / max(shape))).to_vec()
    if turned:  # about y: the detector's v along x
        pg = ts.rotate(pos=0, axis=(0, 1, 0), angles=np.pi / 2) * pg
    return vg, pg


CASES = {
    # 228 MiB of refined projections before the flat kernels' workspace
    "refined": (dict(shape=(64, 64, 64), det=(64, 96), angles=1080), 3, FP),
    # the turned volume and the sums of 64 angles after the swapped volume
    "turned": (dict(shape=(60, 300, 300), det=(300, 3000), angles=70, turned=True), 1, FP),
    # sums beyond the buffer: a long z, many columns
    "wide": (dict(shape=(3000, 40, 40), det=(3000, 350), angles=100), 1, FP),
    # lines of 168 slices where the detector has 146 rows, beside the swapped volume
    "turned_back": (dict(shape=(168, 168, 168), det=(146, 240), angles=1600, turned=True), 1, BP),
}


@pytest.mark.parametrize("case", list(CASES))
def test_noalloc_takes_what_the_padded_and_separable_kernels_fit(monkeypatch, case):
    scan, ss, op = CASES[case]
    A = ts.operator(*_scan(**scan), detector_supersampling=ss)
    plan, lib = A.projector.plan(0), _tsx.load()
    stream = torch.cuda.current_stream().cuda_stream
    # (these variables put the plan on the padded and the separable kernels)
    monkeypatch.setenv("TSX_FP_VARIANT", "4")
    monkeypatch.setenv("TSX_BP_BRICK_Z", "32")
    without = plan.workspace_size(op)
    monkeypatch.delenv("TSX_FP_VARIANT")
    monkeypatch.delenv("TSX_BP_BRICK_Z")
    print(f"[noalloc flat] {case}: workspace {plan.workspace_size(op)} B, {without} B without the flat kernels",
          flush=True)
    assert without <= _tsx.NOALLOC_SCRATCH_BYTES
    gen = torch.Generator(device=DEV)
    gen.manual_seed(3)
    x = torch.rand(A.domain_shape, generator=gen, device=DEV)
    y = torch.rand(A.range_shape, generator=gen, device=DEV)
    out = []
    for fn in (lib.tsx_direct_fpbp3d, lib.tsx_direct_fpbp3d_noalloc):
        vol, proj = x.clone(), y.clone()
        rc = fn(plan.handle, ctypes.c_void_p(vol.data_ptr()), ctypes.c_void_p(proj.data_ptr()), _tsx.TSX_MODE_SET, op,
                ctypes.c_void_p(stream))
        assert rc == 0, lib.tsx_last_error().decode()
        torch.cuda.synchronize()
        out.append(proj if op == FP else vol)
    assert torch.equal(out[0], out[1])
    # and they are the projections: another kernel's, to FP32 rounding
    monkeypatch.setenv("TSX_FP_VARIANT", "4")
    monkeypatch.setenv("TSX_BP_BRICK_Z", "32")
    other = A(x) if op == FP else A.T(y)
    assert rel_l2(out[0].cpu().numpy(), other.cpu().numpy()) <= 5e-6
