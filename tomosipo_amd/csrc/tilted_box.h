// Boxes of detector pixels of the tilted backprojector (bp_tilted): the pixels
// of one detector axis that lie within `half` of a voxel's position. Plain
// arithmetic, for host and device.
#pragma once

#include <math.h>

#ifdef __HIPCC__
#define TSX_BOX_FN __host__ __device__ __forceinline__
#else
#define TSX_BOX_FN inline
#endif

namespace tsx {

struct PixelRange {
    int lo, hi;  // hi < lo: none
};

// Positions and half-widths up to which the integer form holds: all its terms
// stay below 8 reaches (a thread's voxels lie within 7 half-widths of its
// first) and the pixels of an axis, 2^30, so that no sum of two passes 2^31.
constexpr double TILTED_REACH = 67108864.0;

// (false for a position that is not a number)
TSX_BOX_FN bool tilted_in_reach(double cj, double ci) { return fabs(cj) <= TILTED_REACH && fabs(ci) <= TILTED_REACH; }

// The pixels of an axis of n within reach, relative to pixel j0: left and
// right are the floors of half - p and p + half, p the position relative to j0.
TSX_BOX_FN PixelRange tilted_near_pixels(int j0, int left, int right, int n)
{
    const PixelRange r = {-(left < j0 ? left : j0), right < n - 1 - j0 ? right : n - 1 - j0};
    return r;
}

// The pixels of an axis of n within `half` of position c, any c and half: a
// direction of a parallel scan nearly within the detector's plane has
// positions and half-widths of 1e9 pixels and more.
TSX_BOX_FN PixelRange tilted_pixels(double c, double half, int n)
{
    const double lo = fmax(ceil(c - half), 0.0), hi = fmin(floor(c + half), n - 1.0);
    PixelRange r = {0, -1};
    if (c == c && lo <= hi) {
        r.lo = (int)lo;
        r.hi = (int)hi;
    }
    return r;
}

// Cone beams, |W . N| (W from the source to a voxel, N the detector's normal in
// voxel steps along m, c1, c2) above which up to TILTED_VOXELS voxels along c1
// from it on have c = (|N1| + |N2|) / |W . N| <= 1 / 16, the last ones too.
constexpr int TILTED_VOXELS = 8;

TSX_BOX_FN double tilted_apart(const double *N)
{
    return 16.0 * (fabs(N[0]) + fabs(N[1]) + fabs(N[2])) + (TILTED_VOXELS - 1) * fabs(N[1]);
}

// 1 / (1 - c) or a little more, for c <= 1 / 16 (it holds up to 1 / 11).
TSX_BOX_FN float tilted_growth(float c) { return fmaf(1.1f, c, 1.0f); }

}  // namespace tsx
