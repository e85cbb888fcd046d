"""FDK of a large scan's region of interest on the GPU: 2^29 pixels and more.

The upright backprojector takes scans of any number of angles: it addresses the
filtered projections angle by angle. A few voxels around the centre, whose
result differs from the general FDK backprojector's by the rounding of pixel
positions only: 1e-5 of the norm, as between the upright kernel and the oracle.
The workspace is one float per pixel, and less is refused.
"""
import ctypes

import pytest

import tomosipo_amd as ts
from tests.conftest import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_large_upright_scan_takes_the_upright_backprojector(monkeypatch):
    n, angles, roi = 1024, 516, 20
    vg = ts.volume(shape=(roi, roi, roi), size=roi / n)
    pg = ts.cone(angles=angles, shape=(n, n), size=(1.0, 1.0), cone_angle=0.4)
    A = ts.operator(vg, pg)
    plan = A.projector.plan(0)
    assert plan.fdk_workspace_size() == n * n * angles * 4
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    y = torch.rand(A.range_shape, generator=gen, device="cuda")
    ws = torch.empty(n * n * angles, device="cuda")
    out = torch.empty(A.domain_shape, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    with pytest.raises(Exception, match="workspace"):
        plan.fdk(out.data_ptr(), y.data_ptr(), False, s, ctypes.c_void_p(ws.data_ptr()), ws.numel() * 4 - 4)
    plan.fdk(out.data_ptr(), y.data_ptr(), False, s, ctypes.c_void_p(ws.data_ptr()), ws.numel() * 4)
    monkeypatch.setenv("TSX_FORCE_GENERAL", "1")
    general = ts.fdk(A, y)
    assert torch.isfinite(out).all() and not torch.equal(out, general)  # (the other kernel's bits)
    assert rel_l2(out.cpu().numpy(), general.cpu().numpy()) <= 1e-5
