// FDK reconstruction kernels (included by tsx.hip); cone-beam plans only.
//
// fdk_filter: one block per angle and 16 detector rows. The rows are weighted
//   by the cosine of each pixel's ray against the detector normal and convolved
//   on the matrix cores (FP32) with the sampled Ram-Lak kernel g[0] = 1/4,
//   g[odd m] = -1/(pi^2 m^2) over every lag of the row (the linear
//   convolution of the zero-padded row), scaled by 1 / |U|.
// fdk_bp: one thread per voxel; for every angle the voxel centre is projected
//   from the source onto the virtual detector (FP64), the filtered
//   projections are interpolated bilinearly (zero outside) and accumulated
//   with weight (dbeta / 2) * lambda^2, lambda = D / ((X - s) . n).
#pragma once

#include "tsx_plan.h"
#include "fp_kernels.h"

namespace tsx {

constexpr int FDK_MAX_COLS = 4096;
constexpr int FDK_BX = 64, FDK_BY = 4;

// fdk_filter<NT> computes 64 NT outputs of 16 rows in a pass, wave w those of
// parity w & 1 in NT tiles of 16, from 64 NT columns at a time in LDS.
constexpr int FDK_ROWS = 16, FDK_FILTER_THREADS = 256;

// Tiles per wave: the multiplications are passes^2 NT^2, and the loading and
// weighting of the columns for each of passes^2 parts about 5 NT of them.
__host__ __device__ inline int fdk_tiles(int cols)
{
    int best = 12, least = 1 << 30;
    for (int nt = 12; nt >= 2; nt = nt > 8 ? 8 : nt / 2) {
        const int passes = (cols + 64 * nt - 1) / (64 * nt), cost = passes * passes * nt * (nt + 5);
        if (cost < least) {
            least = cost;
            best = nt;
        }
    }
    return best;
}
// Entries of the factor tables on either side of lag 0.
__host__ __device__ inline int fdk_factor_reach(int cols)
{
    const int half = 32 * fdk_tiles(cols);
    return ((cols + 1) / 2 + half - 1) / half * half + 16;
}
constexpr int fdk_filter_floats(int nt) { return 2 * (FDK_ROWS * (32 * nt + 4) + 16) + 64 * nt + 16; }

// q is written as [row][angle][column], or by_angle as [angle][row][column].
//
// The ramp filter couples columns of opposite parity only. With c_p[y] the
// weighted pixel 2 y + p, and E[y] = c_p[y] - c_p[y - 1] the differences of
// the other parity p's pixels (zeros outside the row),
//   q[j] = (2 c[j] - c[j - 1] - c[j + 1]) / 8 + sum_y F(y - j / 2 - (j & 1)) E[y],
//   F(t) = -sign(t) * (sum of 1 / (pi^2 m^2) over the odd m > 2 |t|), F(0) = 0:
// summation by parts of the plain sum, exact because the kernel has no DC
// response. A row that is smooth on the pixel scale has small differences,
// while the terms of the plain sum nearly cancel c[j] / 4. Where a pixel of
// the rows is infinite or NaN, the block takes the plain sum, q[j] = c[j] / 4
// + sum_y H(y - j / 2 - (j & 1)) c_p[y - 1], H(t) = -1 / (pi^2 (2 t - 1)^2),
// which spreads it as the filter's definition says.
//
// Either sum is a product of 16 rows with a Toeplitz matrix: MFMA 16x16x4 in
// FP32, A = the rows (lane: row lane % 16, the slots 4 (lane / 16) + s, s = 0 ..
// 3, of each 16 as one 16-byte LDS read), B = the factors, read from the
// 64 NT + 16 of them that the pass and columns at hand meet. Rows S = 32 NT + 4
// floats apart keep both reads free of bank conflicts; the results go through
// LDS to be written in rows.
//
// Bound: the phases of a block, which loads and weights its rows (an FP64 square
// root per pixel), multiplies (cols FLOP per output, half of the full product: 1.4
// ms of the 3.0 below at the matrix cores' 157 TFLOP/s in FP32) and stores;
// three blocks per CU at 768 columns, so that one loads while another
// multiplies. 512 x 720 rows of 768 columns: 3.0 ms (the sum
// of factor (c[j - m] + c[j + m] - 2 c[j]) on the vector ALUs, register-tiled:
// 10.4 ms; in this form there: 9.5 ms).
template <int NT>
__global__ void __launch_bounds__(FDK_FILTER_THREADS, NT > 8 ? 3 : 4)
fdk_filter(const FdkAngle *__restrict__ angles, int n_angles, int rows, int cols, const float *__restrict__ factors,
           const float *__restrict__ proj, float *__restrict__ q, int by_angle)
{
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int HALF = 32 * NT, S = HALF + 4, PAR = FDK_ROWS * S + 16, W = 2 * HALF + 4, OUT = 2 * HALF + 4;
    __shared__ __align__(16) float lds[fdk_filter_floats(NT)];
    float *tab = lds + 2 * PAR;
    const int i0 = blockIdx.x * FDK_ROWS, a = blockIdx.y;
    const FdkAngle &A = angles[a];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = wave & 1, u0 = (wave >> 1) * 16 * NT, n = lane & 15, h = lane >> 4;
    const int passes = ((cols + 1) / 2 + HALF - 1) / HALF;
    const int64_t pitch = (int64_t)n_angles * cols;
    const float *src = proj + (int64_t)i0 * pitch + (int64_t)a * cols;
    int plain = 0;
    if (passes > 1) {  // every pass and every part of a row has to take the same sum
        bool bad = false;
        for (int r = 0; r < FDK_ROWS && i0 + r < rows; ++r)
            for (int k = threadIdx.x; k < cols; k += FDK_FILTER_THREADS)
                bad |= !(fabsf(src[r * pitch + k]) <= 3.402823466e38f);
        plain = __syncthreads_or(bad);
    }
    for (int pass = 0; pass < passes; ++pass) {
        const int ub = pass * HALF;
        f4 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int k = 0; k < passes; ++k) {
            // (the pass's own columns come last: the outputs need them)
            const int part = (pass + 1 + k) % passes, yb = part * HALF;
            // slot s of row r and parity p: c_p[yb - 1 + s], s = 0 .. HALF + 1
            bool bad = false;
            __syncthreads();
#pragma unroll 2
            for (int e = threadIdx.x; e < FDK_ROWS * W; e += FDK_FILTER_THREADS) {
                const int r = e / W, kk = e - r * W, j = 2 * yb - 2 + kk, i = i0 + r;
                float v = 0.0f;
                if (j >= 0 && j < cols && i < rows) {
                    const double px = A.P0s[0] + j * A.U[0] + i * A.V[0];
                    const double py = A.P0s[1] + j * A.U[1] + i * A.V[1];
                    const double pz = A.P0s[2] + j * A.U[2] + i * A.V[2];
                    v = (float)(A.D / sqrt(px * px + py * py + pz * pz) * (double)src[r * pitch + j]);
                }
                bad |= !(fabsf(v) <= 3.402823466e38f);
                lds[(kk & 1) * PAR + r * S + (kk >> 1)] = v;
            }
            plain |= __syncthreads_or(bad);
            const int reach = passes * HALF + 16;
            const float *f = factors + (plain ? 2 * reach + 1 : 0) + reach + (yb - ub) - HALF;
            for (int e = threadIdx.x; e < 2 * HALF + 16; e += FDK_FILTER_THREADS) tab[e] = f[e];
            __syncthreads();
            // the other parity's differences (or pixels) yb .. yb + nd - 1
            const int nd = part == passes - 1 ? (p ? (cols + 1) / 2 : cols / 2) + 1 - yb : HALF;
            const float *line = lds + (1 - p) * PAR + n * S + 4 * h;
            const float *fac = tab + HALF - u0 - p + 4 * h - n;
            for (int kb = 0; kb < nd; kb += 16) {
                const float4 c = *reinterpret_cast<const float4 *>(line + kb);
                const float next = line[kb + 4];
                float e[4];
                e[0] = plain ? c.x : c.y - c.x;
                e[1] = plain ? c.y : c.z - c.y;
                e[2] = plain ? c.z : c.w - c.z;
                e[3] = plain ? c.w : next - c.w;
                if (kb + 16 > nd) {
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        if (kb + 4 * h + s >= nd) e[s] = 0.0f;
                }
#pragma unroll
                for (int s = 0; s < 4; ++s) {
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(e[s], fac[kb - 16 * t + s], acc[t], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // acc[t][g]: row 4 h + g, column 2 (ub + u0 + 16 t + n) + p
        const float inv_du = (float)A.inv_du;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int u = u0 + 16 * t + n;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float *even = lds + (4 * h + g) * S + u, *odd = even + PAR;
                const float c = p ? odd[1] : even[1], l = p ? even[1] : odd[0], r = p ? even[2] : odd[1];
                acc[t][g] = inv_du * (plain ? fmaf(0.25f, c, acc[t][g]) : fmaf(0.125f, (c - l) + (c - r), acc[t][g]));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g) lds[(4 * h + g) * OUT + 2 * (u0 + 16 * t + n) + p] = acc[t][g];
        __syncthreads();
        for (int e = threadIdx.x; e < FDK_ROWS * 2 * HALF; e += FDK_FILTER_THREADS) {
            const int r = e / (2 * HALF), k = e - r * 2 * HALF, j = 2 * ub + k, i = i0 + r;
            if (j >= cols || i >= rows) continue;
            const float v = lds[r * OUT + k];
            q[by_angle ? ((int64_t)a * rows + i) * cols + j : (int64_t)i * pitch + (int64_t)a * cols + j] = v;
        }
    }
}

__global__ void __launch_bounds__(FDK_BX *FDK_BY)
fdk_bp(const FdkAngle *__restrict__ angles, int n_angles, int rows, int cols,
       const float *__restrict__ q, float *__restrict__ vol, int nx, int ny, int nz, double lo_x,
       double lo_y, double lo_z, double h_x, double h_y, double h_z, int additive)
{
    const int x = blockIdx.x * FDK_BX + threadIdx.x;
    const int y = blockIdx.y * FDK_BY + threadIdx.y;
    const int z = blockIdx.z;
    if (x >= nx || y >= ny) return;
    const double X = lo_x + (x + 0.5) * h_x, Y = lo_y + (y + 0.5) * h_y, Z = lo_z + (z + 0.5) * h_z;
    const int64_t astride = cols, rstride = (int64_t)n_angles * cols;
    float acc = 0.0f;
    for (int a = 0; a < n_angles; ++a) {
        const FdkAngle &A = angles[a];
        const double wx = X - A.s[0], wy = Y - A.s[1], wz = Z - A.s[2];
        const double den = wx * A.n[0] + wy * A.n[1] + wz * A.n[2];
        if (!(den > 0.0)) continue;  // voxel not in front of the source
        const double lam = A.D * rcp64(den);
        const double fj = A.cj + lam * (wx * A.Bj[0] + wy * A.Bj[1] + wz * A.Bj[2]);
        const double fi = A.ci + lam * (wx * A.Bi[0] + wy * A.Bi[1] + wz * A.Bi[2]);
        if (!(fj > -1.0 && fj < (double)cols && fi > -1.0 && fi < (double)rows)) continue;
        const double fj0 = floor(fj), fi0 = floor(fi);
        const int j0 = (int)fj0, i0 = (int)fi0;
        const float wj = (float)(fj - fj0), wi = (float)(fi - fi0);
        // corners outside the detector read a clamped (in-bounds) pixel and count 0
        const float *base = q + (int64_t)a * astride;
        const bool j_lo = j0 >= 0, j_hi = j0 + 1 < cols, i_lo = i0 >= 0, i_hi = i0 + 1 < rows;
        const int jc0 = max(j0, 0), jc1 = min(j0 + 1, cols - 1);
        const int64_t r0 = (int64_t)max(i0, 0) * rstride, r1 = (int64_t)min(i0 + 1, rows - 1) * rstride;
        const float v00 = (i_lo && j_lo) ? base[r0 + jc0] : 0.0f;
        const float v01 = (i_lo && j_hi) ? base[r0 + jc1] : 0.0f;
        const float v10 = (i_hi && j_lo) ? base[r1 + jc0] : 0.0f;
        const float v11 = (i_hi && j_hi) ? base[r1 + jc1] : 0.0f;
        const float lo = fmaf(wj, v01 - v00, v00);
        const float hi = fmaf(wj, v11 - v10, v10);
        acc = fmaf((float)(A.half_dbeta * lam * lam), fmaf(wi, hi - lo, lo), acc);
    }
    float *o = vol + ((int64_t)z * ny + y) * nx + x;
    *o = additive ? *o + acc : acc;
}

// Upright detectors (v parallel to z, detector normal perpendicular to z, every
// angle; q as [angle][row][column]): along a voxel column (x, y) the depth, the
// detector column and the weight are constant and the detector row is affine
// in z. A block takes 16 x 16 columns and ZC voxels of each: FP64 setup
// once per column and angle, FP32 per voxel.
//
// The pixels that the block's voxels read at an angle lie between those of its
// corners (formed for eight angles at a time, a corner per lane); they are
// staged in LDS with zeros around the detector, the next angle's while the
// present one's are summed (two buffers, one barrier per angle). Where they
// are more than the buffer holds (pixels far finer than the voxels) or a
// corner is not in front of the source, the angle's pixels are read from
// memory, each with its own bounds.
//
// Bound: vector ALU issue (1.06 instructions per CU-cycle: 12 per voxel and
// angle and the setup), with 0.14 LDS reads (two of 8 bytes per voxel and
// angle) beside it. A 16-byte gather from row-paired memory
// took 16 cycles of the L1 port per wave: 512^3, 720 angles, 512 x 768
// pixels 49.0 ms; 39.7 ms so.
//
// ZC voxels per column; staged are at most SP columns (the pitch) and SR rows.
// 32 voxels share a set-up better than 16 (39.7 and 42.0 ms); detectors with
// pixels finer than about a voxel take 8 and larger pieces.
constexpr int FDK_T = 16;

template <int ZC, int SP, int SR>
__global__ void __launch_bounds__(FDK_T *FDK_T)
fdk_bp_upright(const FdkAngle *__restrict__ angles, int n_angles, int rows, int cols,
               const float *__restrict__ q, float *__restrict__ vol, int nx, int ny, int nz,
               double lo_x, double lo_y, double lo_z, double h_x, double h_y, double h_z, int additive)
{
    constexpr int THREADS = FDK_T * FDK_T, LOADS = (SP * SR + THREADS - 1) / THREADS;
    __shared__ float pixels[2][LOADS * THREADS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int x0 = blockIdx.x * FDK_T, y0 = blockIdx.y * FDK_T, z0 = blockIdx.z * ZC;
    const int x = x0 + (tid & (FDK_T - 1)), y = y0 + tid / FDK_T;
    // (threads past the volume repeat its last column: positions stay between the corners')
    const double X = lo_x + (min(x, nx - 1) + 0.5) * h_x, Y = lo_y + (min(y, ny - 1) + 0.5) * h_y;
    const double Z0 = lo_z + (z0 + 0.5) * h_z;
    float acc[ZC];
#pragma unroll
    for (int k = 0; k < ZC; ++k) acc[k] = 0.0f;
    // lane 8 e + c: corner c of the block at angle a0 + e, then the angle's first
    // staged column and row and their numbers (0 columns: not staged)
    int first_j = 0, first_i = 0, wide = 0, high = 0;
    auto corners = [&](int a0) {
        const FdkAngle &A = angles[min(a0 + (lane >> 3), n_angles - 1)];
        const double cx = lo_x + (x0 + (lane & 1 ? FDK_T - 1 : 0) + 0.5) * h_x;
        const double cy = lo_y + (y0 + (lane & 2 ? FDK_T - 1 : 0) + 0.5) * h_y;
        const double cz = lo_z + (z0 + (lane & 4 ? ZC - 1 : 0) + 0.5) * h_z;
        const double wx = cx - A.s[0], wy = cy - A.s[1], wz = cz - A.s[2];
        const double den = wx * A.n[0] + wy * A.n[1];
        int bad = !(den > 1e-6 * A.D);
        const double lam = bad ? 0.0 : A.D / den;
        double j_lo = A.cj + lam * (wx * A.Bj[0] + wy * A.Bj[1]);
        double i_lo = A.ci + lam * (wx * A.Bi[0] + wy * A.Bi[1] + wz * A.Bi[2]);
        double j_hi = j_lo, i_hi = i_lo;
#pragma unroll
        for (int d = 1; d < 8; d *= 2) {
            j_lo = fmin(j_lo, __shfl_xor(j_lo, d, 64));
            j_hi = fmax(j_hi, __shfl_xor(j_hi, d, 64));
            i_lo = fmin(i_lo, __shfl_xor(i_lo, d, 64));
            i_hi = fmax(i_hi, __shfl_xor(i_hi, d, 64));
            bad |= __shfl_xor(bad, d, 64);
        }
        // (the margins exceed the rounding of the voxels' positions, FP64 and FP32)
        bad |= !(j_hi - j_lo < SP - 3.0 && i_hi - i_lo < SR - 3.0 && fabs(j_lo) < 1e8 && fabs(i_lo) < 1e8);
        first_j = bad ? 0 : (int)floor(j_lo - 1e-6);
        first_i = bad ? 0 : (int)floor(i_lo - 1e-3);
        wide = bad ? 0 : (int)floor(j_hi + 1e-6) + 2 - first_j;
        high = bad ? 0 : (int)floor(i_hi + 1e-3) + 2 - first_i;
    };
    float next[LOADS];
    int count = 0;
    // pixel e = (row e / SP, column e % SP) of the staged ones of angle a
    auto load = [&](int a) {
        const int e8 = (a & 7) * 8;
        const int fj = __builtin_amdgcn_readlane(first_j, e8), fi = __builtin_amdgcn_readlane(first_i, e8);
        const int w = __builtin_amdgcn_readlane(wide, e8), h = __builtin_amdgcn_readlane(high, e8);
        const float *src = q + (int64_t)a * rows * cols;
        count = w ? h * SP : 0;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            if (l * THREADS >= count) break;
            const int e = l * THREADS + tid, r = e / SP, c = e - r * SP, i = fi + r, j = fj + c;
            next[l] = 0.0f;
            if (c < w && (unsigned)i < (unsigned)rows && (unsigned)j < (unsigned)cols) next[l] = src[i * cols + j];
        }
    };
    corners(0);
    load(0);
    for (int a = 0; a < n_angles; ++a) {
        float *buf = pixels[a & 1];
        const int e8 = (a & 7) * 8;
        const bool staged = __builtin_amdgcn_readlane(wide, e8) > 0;
        const int fj0 = __builtin_amdgcn_readlane(first_j, e8), fi0 = __builtin_amdgcn_readlane(first_i, e8);
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {
            if (l * THREADS >= count) break;
            buf[l * THREADS + tid] = next[l];
        }
        __syncthreads();
        if (a + 1 < n_angles) {
            if (((a + 1) & 7) == 0) corners(a + 1);
            load(a + 1);
        }
        const FdkAngle &A = angles[a];
        const double wx = X - A.s[0], wy = Y - A.s[1], wz = Z0 - A.s[2];
        const double den = wx * A.n[0] + wy * A.n[1];
        const double lam = A.D * rcp64(den);
        const double fj = A.cj + lam * (wx * A.Bj[0] + wy * A.Bj[1]) - fj0;
        const double fi = A.ci + lam * (wx * A.Bi[0] + wy * A.Bi[1] + wz * A.Bi[2]) - fi0;
        const float dfi = (float)(lam * h_z * A.Bi[2]), wgt = (float)(A.half_dbeta * lam * lam);
        if (staged) {
            const double fl = floor(fj);
            const float cb = (float)(fj - fl), ca = 1.0f - cb, f0 = (float)fi;
            const float *col = buf + (int)fl;
#pragma unroll
            for (int k = 0; k < ZC; ++k) {
                const float f = fmaf((float)k, dfi, f0), ff = floorf(f), wi = f - ff;
                const float *p = col + (int)__umul24((uint32_t)(int)ff, SP);
                const float top = fmaf(ca, p[0], cb * p[1]), bot = fmaf(ca, p[SP], cb * p[SP + 1]);
                acc[k] = fmaf(wgt, fmaf(wi, bot - top, top), acc[k]);
            }
        } else if (x < nx && y < ny && den > 0.0 && fj > -1.0 && fj < (double)cols) {
            const double fl = floor(fj);
            const int j0 = (int)fl;
            const float wj = (float)(fj - fl);
            const float *src = q + (int64_t)a * rows * cols;
            const bool j_lo = j0 >= 0, j_hi = j0 + 1 < cols;
            const double step = lam * h_z * A.Bi[2];
            for (int k = 0; k < ZC; ++k) {
                const double f = fma((double)k, step, fi), ff = floor(f);
                if (!(f > -1.0 && f < (double)rows)) continue;
                const int i0 = (int)ff;
                const float wi = (float)(f - ff);
                const float *r0 = src + (int64_t)i0 * cols + j0, *r1 = r0 + cols;
                const bool i_lo = i0 >= 0, i_hi = i0 + 1 < rows;
                const float v00 = (i_lo && j_lo) ? r0[0] : 0.0f, v01 = (i_lo && j_hi) ? r0[1] : 0.0f;
                const float v10 = (i_hi && j_lo) ? r1[0] : 0.0f, v11 = (i_hi && j_hi) ? r1[1] : 0.0f;
                const float top = fmaf(1.0f - wj, v00, wj * v01), bot = fmaf(1.0f - wj, v10, wj * v11);
                const float t = wgt * fmaf(wi, bot - top, top);
#pragma unroll
                for (int e = 0; e < ZC; ++e)
                    if (e == k) acc[e] += t;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < ZC; ++k) {
        const int z = z0 + k;
        if (x < nx && y < ny && z < nz) {
            float *o = vol + ((int64_t)z * ny + y) * nx + x;
            *o = additive ? *o + acc[k] : acc[k];
        }
    }
}

using FdkKernel = void (*)(const FdkAngle *, int, int, int, const float *, float *, int, int, int, double, double, double,
                           double, double, double, int);
constexpr int FDK_ZC = 32, FDK_SP = 41, FDK_SR = 62, FDK_FINE_ZC = 8, FDK_FINE_SP = 83, FDK_FINE_SR = 58;

}  // namespace tsx
