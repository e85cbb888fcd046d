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

// With `pair`, q is written row-paired: element (i, a, j) holds the filtered
// values of rows i and i + 1 (0 past the last row), 8 bytes.
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
// Bound: the matrix cores' FP32 rate (157 TFLOP/s; 2 cols FLOP per output,
// half of the full product), with three blocks per CU at 768 columns so that
// one loads while another multiplies. 512 x 720 rows of 768 columns: FIGURE ms (the sum
// of factor (c[j - m] + c[j + m] - 2 c[j]) on the vector ALUs, register-tiled:
// 10.4 ms; in this form there: 9.5 ms).
template <int NT>
__global__ void __launch_bounds__(FDK_FILTER_THREADS, NT > 8 ? 3 : 4)
fdk_filter(const FdkAngle *__restrict__ angles, int n_angles, int rows, int cols, const float *__restrict__ factors,
           const float *__restrict__ proj, float *__restrict__ q, int pair)
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
            const int64_t o = (int64_t)i * pitch + (int64_t)a * cols + j;
            if (!pair) {
                q[o] = v;
            } else {
                if (i == rows - 1)
                    reinterpret_cast<float2 *>(q)[o] = make_float2(v, 0.0f);
                else if (r < FDK_ROWS - 1)
                    reinterpret_cast<float2 *>(q)[o] = make_float2(v, lds[(r + 1) * OUT + k]);
                else
                    q[2 * o] = v;
                if (r == 0 && i > 0) q[2 * (o - pitch) + 1] = v;
            }
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
// angle; at least 2 detector columns; row-paired q): along a voxel column (x, y) the depth,
// the detector column and the weight are constant and the detector row is
// affine in z. One thread per (x, y) and FDK_ZC voxels along z: FP64 setup
// once per angle, FP32 per voxel; the waves of a block go through the angles
// in step (a barrier per angle).
constexpr int FDK_ZC = 16;

__global__ void __launch_bounds__(FDK_BX *FDK_BY)
fdk_bp_upright(const FdkAngle *__restrict__ angles, int n_angles, int rows, int cols,
               const float *__restrict__ q, float *__restrict__ vol, int nx, int ny, int nz,
               double lo_x, double lo_y, double lo_z, double h_x, double h_y, double h_z, int additive)
{
    const int x = blockIdx.x * FDK_BX + threadIdx.x;
    const int y = blockIdx.y * FDK_BY + threadIdx.y;
    const int z0 = blockIdx.z * FDK_ZC;
    const bool active = x < nx && y < ny;  // every thread takes part in the barriers
    const double X = lo_x + (x + 0.5) * h_x, Y = lo_y + (y + 0.5) * h_y, Z0 = lo_z + (z0 + 0.5) * h_z;
    // the row-paired filtered projections are addressed with 32-bit byte offsets (< 4 GiB)
    const uint32_t rbytes = (uint32_t)n_angles * (uint32_t)cols * 8u;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)q, (short)0, (int)(rbytes * (uint32_t)rows), 0x00020000);
    float acc[FDK_ZC];
#pragma unroll
    for (int k = 0; k < FDK_ZC; ++k) acc[k] = 0.0f;
    for (int a = 0; a < n_angles; ++a) {
        auto one_angle = [&]() {
            const FdkAngle &A = angles[a];
            const double wx = X - A.s[0], wy = Y - A.s[1], wz = Z0 - A.s[2];
            const double den = wx * A.n[0] + wy * A.n[1];
            if (!(den > 0.0)) return;
            const double lam = A.D * rcp64(den);
            const double fj = A.cj + lam * (wx * A.Bj[0] + wy * A.Bj[1]);
            if (!(fj > -1.0 && fj < (double)cols)) return;
            // rows relative to the first voxel's, floor(fi): FP32 holds their fractions
            const double fi = fmin(fmax(A.ci + lam * (wx * A.Bi[0] + wy * A.Bi[1] + wz * A.Bi[2]), -1e9), 1e9);
            const int ib = (int)floor(fi);
            const float fi0 = (float)(fi - ib);
            const float dfi = (float)(lam * h_z * A.Bi[2]);
            const float wgt = (float)(A.half_dbeta * lam * lam);
            const double fj0 = floor(fj);
            const int j0 = (int)fj0;
            const float wj = (float)(fj - fj0);
            // columns (jb, jb + 1), jb = j0 clamped into [0, cols - 2], read as one
            // 8-byte pair; the weights of columns outside the detector are 0
            const int jb = min(max(j0, 0), max(cols - 2, 0));
            float ca, cb;
            if (j0 == jb) {
                ca = 1.0f - wj;
                cb = j0 + 1 < cols ? wj : 0.0f;
            } else if (j0 < jb) {  // j0 = -1: only column 0 = jb, weight wj
                ca = wj;
                cb = 0.0f;
            } else {               // j0 = cols - 1: only column jb + 1, weight 1 - wj
                ca = 0.0f;
                cb = 1.0f - wj;
            }
            // q is row-paired: the 16 bytes at (row i, column jb) are
            // q[i][jb], q[i+1][jb], q[i][jb+1], q[i+1][jb+1]
            const uint32_t cboff = ((uint32_t)a * (uint32_t)cols + (uint32_t)jb) * 8u;
    #pragma unroll
            for (int k = 0; k < FDK_ZC; ++k) {
                const float fi = fmaf((float)k, dfi, fi0);
                const float fi0f = floorf(fi);
                const int i0 = ib + (int)fi0f;
                const float wi = fi - fi0f;
                // rows i0, i0 + 1 from the element of row max(i0, 0) (inside the
                // buffer); for i0 = -1 that element's first row is row i0 + 1
                const uint32_t o = (uint32_t)min(max(i0, 0), rows - 1) * rbytes + cboff;
                const float x0 = bload(rs, o), y0 = bload(rs, o + 4u);
                const float x1 = bload(rs, o + 8u), y1 = bload(rs, o + 12u);
                const float first = fmaf(ca, x0, cb * x1), second = fmaf(ca, y0, cb * y1);
                const bool in = i0 >= 0 && i0 < rows;
                const float top = in ? first : 0.0f;
                const float bot = in ? second : (i0 == -1 ? first : 0.0f);
                acc[k] = fmaf(wgt, fmaf(wi, bot - top, top), acc[k]);
            }
        };
        if (active) one_angle();
        // The block's waves stay at one angle together: their voxels read
        // neighbouring pixels of the same filtered projection, which the
        // waves then share in L1 (17 % faster at 512^3 than free-running).
        __syncthreads();

    }
#pragma unroll
    for (int k = 0; k < FDK_ZC; ++k) {
        const int z = z0 + k;
        if (active && z < nz) {
            float *o = vol + ((int64_t)z * ny + y) * nx + x;
            *o = additive ? *o + acc[k] : acc[k];
        }
    }
}

}  // namespace tsx
