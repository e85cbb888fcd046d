"""Which plans run on the flat kernels, as tsx_plan_info says (host plans, no GPU)."""
import ctypes

import numpy as np
import pytest

import tomosipo_amd as ts
from tomosipo_amd import _tsx


def _info(vg, pg, **options):
    return ts.operator(vg, pg, **options).projector._host_plan.info()


def test_info_names_the_flat_kernels(monkeypatch):
    vg = ts.volume(shape=(40, 48, 56), size=(40 / 48, 1, 56 / 48))
    par = ts.parallel(angles=20, shape=(40, 72), size=(1, 1.5)).to_vec()
    cone = ts.cone(angles=20, shape=(40, 72), size=(1, 1.5), cone_angle=0.5).to_vec()
    turned = ts.rotate(pos=0, axis=(0, 1, 0), angles=np.pi / 2) * par
    tilted = ts.rotate(pos=0, axis=(0, 1, 0), angles=0.2) * par
    for pg, options, flat in ((par, {}, True), (cone, {}, False), (turned, {}, True), (tilted, {}, False),
                              (par, {"detector_supersampling": 2}, True), (cone, {"detector_supersampling": 2}, False)):
        info = _info(vg, pg, **options)
        assert (info["fp_flat"], info["bp_flat"]) == (flat, flat), (options, info)
    # pixels finer than half a voxel keep the separable backprojector
    fine = ts.parallel(angles=20, shape=(40, 300), size=(1, 1.5))
    info = _info(vg, fine)
    assert info["fp_flat"] and not info["bp_flat"] and info["bp_kernel"] == "separable"
    # a variable that asks for one of the other kernels' forms
    monkeypatch.setenv("TSX_FP_VARIANT", "4")
    assert not _info(vg, par)["fp_flat"] and _info(vg, par)["bp_flat"]
    monkeypatch.setenv("TSX_BP_BRICK_Z", "24")
    assert not _info(vg, par)["bp_flat"]


def test_info_keeps_the_size_of_its_structure():
    assert ctypes.sizeof(_tsx.TsxPlanInfo) == 120
