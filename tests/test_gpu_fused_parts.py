"""Fused backprojections of instances whose angles are summed in parts (GPU).

The parts run in separate blocks or in turn, whichever the launch's bricks
make faster; every instance equals its own call bitwise either way, with each
epilogue and in calls of more instances than a launch holds.
"""
import numpy as np
import pytest

import tomosipo_amd as ts

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _cone(n, angles):
    vg = ts.volume(shape=(n, n, n + 3), size=1)
    return ts.operator(vg, ts.cone(angles=angles, shape=(n, 3 * n // 2), size=(1.4, 2.1), cone_angle=0.5))


CASES = {
    "apart": [(48, 40), (33, 17), (20, 9)],
    "in_turn": [(64, 24)] * 16,
    "two_launches": [(20 + k, 30 - k) for k in range(19)],
    "one": [(40, 50)],
    "with_one_part": [(32, 3), (32, 40), (24, 4)],
}


@pytest.mark.parametrize("case", list(CASES))
def test_fused_parts_equal_single_calls(case):
    from tomosipo_amd.fused import Epilogue, fused_backward

    ops = [_cone(n, a) for n, a in CASES[case]]
    gen = torch.Generator(device=DEV)
    gen.manual_seed(6)
    ys = [torch.randn(A.range_shape, generator=gen, device=DEV) for A in ops]
    cs = [torch.rand(A.domain_shape, generator=gen, device=DEV) for A in ops]
    xs = [torch.randn(A.domain_shape, generator=gen, device=DEV) for A in ops]
    want = [A.T(y) for A, y in zip(ops, ys)]
    for got, b in zip(fused_backward(ops, ys), want):
        assert torch.equal(got, b)
    outs = fused_backward(ops, ys, out=[x.clone() for x in xs], epilogues=[Epilogue("add")] * len(ops))
    for got, b, x in zip(outs, want, xs):
        assert torch.equal(got, x + b)
    outs = fused_backward(ops, ys, out=[x.clone() for x in xs],
                          epilogues=[Epilogue("scaled_add", w=c) for c in cs])
    for got, b, x, c in zip(outs, want, xs, cs):
        assert np.linalg.norm((got - (x + c * b)).cpu().numpy()) <= 1e-6 * np.linalg.norm((x + c * b).cpu().numpy())
