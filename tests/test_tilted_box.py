"""The pixel boxes of the tilted backprojector (csrc/tilted_box.h) on the CPU.

A parallel scan with a direction nearly within its detector's plane is
accepted: voxels then map 1e9 pixels and more beyond the detector, and so
large are the images of their squares. Whatever the position, a box is the
detector's pixels within the half-width, or empty; a box that came out larger
than the detector is a loop that does not end.
"""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tomosipo_amd", "csrc")

SHIM = r"""
#include <limits.h>
#include "tilted_box.h"
using namespace tsx;
// (as the hardware converts: saturating, 0 for what is no number)
static int floor_to_int(float v)
{
    v = floorf(v);
    return v != v ? 0 : v >= 2147483648.0f ? INT_MAX : v < -2147483648.0f ? INT_MIN : (int)v;
}
extern "C" void far_box(double c, float half, int n, int *out)
{
    const PixelRange r = tilted_pixels(c, half, n);
    out[0] = r.lo;
    out[1] = r.hi;
}
// voxel k of a thread whose first one is at c, steps apart; 0 where the kernel takes the other form
extern "C" int near_box(double c, float step, int k, float half, int n, int *out)
{
    const float reach = (float)TILTED_REACH;
    if (!(tilted_in_reach(c, 0.0) && fabsf(step) <= reach && half <= reach)) return 0;
    const int j0 = (int)floor(c);
    const float p = fmaf((float)k, step, (float)(c - j0));
    const PixelRange r = tilted_near_pixels(j0, floor_to_int(half - p), floor_to_int(p + half), n);
    out[0] = r.lo;
    out[1] = r.hi;
    out[2] = j0;
    return 1;
}
extern "C" double apart(const double *N) { return tilted_apart(N); }
extern "C" float growth(float c) { return tilted_growth(c); }
"""


@pytest.fixture(scope="module")
def boxes(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("box")
    (d / "shim.cpp").write_text(SHIM)
    so = str(d / "shim.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ftrapv", "-shared", "-fPIC", "-I", CSRC, "-o", so,
                    str(d / "shim.cpp")], check=True, capture_output=True, timeout=120)
    lib = ctypes.CDLL(so)
    lib.far_box.argtypes = [ctypes.c_double, ctypes.c_float, ctypes.c_int, ctypes.c_void_p]
    lib.near_box.argtypes = [ctypes.c_double, ctypes.c_float, ctypes.c_int, ctypes.c_float, ctypes.c_int,
                             ctypes.c_void_p]
    lib.apart.restype = ctypes.c_double
    lib.apart.argtypes = [ctypes.c_void_p]
    lib.growth.restype = ctypes.c_float
    lib.growth.argtypes = [ctypes.c_float]
    return lib


MAGNITUDES = [0.0, 0.3, 1.0, 7.6, 40.0, 1e3, 3e5, 6e7, 6.7e7, 6.8e7, 1e8, 1e9, 2.1e9, 3.2e9, 5e9, 1e10, 1e12, 1e30]


def _brute(c, half, n):
    j = np.arange(n)
    hit = j[np.abs(j - c) <= half]
    return (int(hit[0]), int(hit[-1])) if len(hit) else None


@pytest.mark.parametrize("n", [1, 2, 48])
def test_boxes_beyond_reach_are_cut_to_the_detector(boxes, n):
    out = (ctypes.c_int * 2)()
    for c in [s * m + o for m in MAGNITUDES for s in (-1, 1) for o in (0.0, 0.25, n - 1)] + [np.nan, np.inf, -np.inf]:
        for half in MAGNITUDES + [np.inf]:
            half = float(np.float32(half))
            boxes.far_box(c, half, n, out)
            lo, hi = out
            if np.isfinite(c):
                want = _brute(c, half, n)
                assert (lo, hi) == want if want else hi < lo, (c, half, n, lo, hi)
            assert hi < lo or 0 <= lo <= hi < n, (c, half, n, lo, hi)


@pytest.mark.parametrize("n", [1, 2, 48, 2 ** 30 - 1])
def test_boxes_within_reach_never_leave_the_detector(boxes, n):
    out = (ctypes.c_int * 3)()
    taken = 0
    for c in [s * m + o for m in MAGNITUDES for s in (-1, 1) for o in (0.0, 0.25, min(n, 99) - 1)] + [np.nan, np.inf]:
        for half in MAGNITUDES + [np.inf]:
            for step in (0.0, 0.7, -3e4, 6e7, -6.7e7, 1e9, -5e9):
                for k in (0, 1, 7):
                    if not boxes.near_box(c, step, k, half, n, out):
                        continue
                    taken += 1
                    lo, hi, j0 = out
                    assert lo + j0 >= 0 and hi + j0 <= n - 1 and hi - lo < n, (c, half, step, k, lo, hi, j0)
                    # (positions of moderate size: the pixels of the FP64 box, but for those at its very edge)
                    if n < 1000 and abs(c) < 1e3 and abs(step) < 1.0 and half < 1e3:
                        for edge, cut in ((1e-3, max), (-1e-3, min)):
                            want = _brute(c + k * float(np.float32(step)), max(0.0, half + edge), n)
                            if want and edge < 0:
                                assert lo + j0 <= want[0] and hi + j0 >= want[1]
                            elif want:
                                assert hi < lo or (lo + j0 >= want[0] and hi + j0 <= want[1])
    assert taken > 1000


def test_box_growth_covers_every_voxel_of_a_thread(boxes):
    """The image of a voxel's square is at most 1 / (1 - c) of its linear part,
    c = (|N1| + |N2|) / |W . N|; the thread's voxels lie k N1 further, k < 8."""
    rng = np.random.default_rng(7)
    normals = np.concatenate([rng.standard_normal((500, 3)), [[0, 1, 0], [0.01, 1, 0.01], [0, 1, 1], [1, 0, 0]]])
    for N in normals:
        N = np.ascontiguousarray(N)
        dn = boxes.apart(N.ctypes.data) * (1 + 1e-6)
        for sign in (1, -1):
            c = (abs(N[1]) + abs(N[2])) / np.abs(sign * dn + np.arange(8) * N[1])
            assert c.max() <= 1 / 16 + 1e-9 and boxes.growth(c.max()) >= 1 / (1 - c.max()), (N, c.max())
