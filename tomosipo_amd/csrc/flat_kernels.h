// Flat parallel-beam kernels (included by tsx.hip): scans whose rays stay
// within a slice of constant z (parallel beam, ray direction perpendicular to
// z, detector v parallel to z, stepping axis x or y at every angle).
//
// There the Joseph weights factor: ray (a, i, j) meets slice n of its stepping
// axis at the in-slice position q(a, j, n), the same for every detector row i,
// and at the height t(a, i, j), the same for every slice. So
//   forward:   G[a, j, z] = sum_n lerp_q x[n, ., z],  y[i, a, j] = l lerp_t G[a, j, .]
//   backward:  U[a, j, z] = sum_i L(t - z) l y[i, a, j],
//              x[n, c, z] = sum_a sum_j L(q(a, j, n) - c) U[a, j, z],
// and the sums over slices and columns have one weight for a whole line along
// z. The kernels keep z contiguous (volume turned to [x][y][w], G and U as
// [angle][column][w]; w = (batch entry, z), so that short stacks and 2D
// slices of a batch fill the lanes), take consecutive w per lane and share the
// weights that one lane formed (through LDS or v_readlane): 2 fma per (ray,
// slice, z) or (voxel, column) instead of a gather and a bilinear
// interpolation of their own.
//
// Every lane's arithmetic and its order depend only on the plan, never on the
// position of its w in a wave, so single, batched and fused launches give
// the same bits.
#pragma once

#include "tsx_plan.h"
#include "fp_kernels.h"
#include "bp_kernels.h"

namespace tsx {

constexpr int FLAT_MAX = MAX_FUSED;  // instances of one launch
constexpr int FLAT_STRIP = 8;        // forward projector: column tiles per strip
// forward: slices (n / FLAT_SUM of the volume) summed before they join the rest of a ray's sum.
// One running sum over the 256 slices of a slice stack rounds to 3.6e-7 of the result, the
// padded kernels' two to 1.9e-7, sums of 32 to 1.6e-7 (for 1 to 2 % of the time).
constexpr int FLAT_SUM = 32;
constexpr int FLAT_BX = 16, FLAT_BY = 8;  // backprojector: voxel columns per brick (one wave per y)
constexpr int FLAT_BSC = 64;         // most detector columns staged per angle

// One instance as seen by the kernels of a launch over the angles
// ang[0 .. kn - 1] of the plan's axis-ordered table.
struct FlatView {
    const FlatAngle *ang;
    int kn;                 // angles of the launch
    int n_angles, rows, cols, nx, ny, nz;
    int W, Wp;              // batch entries x nz, and the pitch of a line
    float *vol, *proj;      // caller's data: read or written, entries vs and ps floats apart
    int64_t vs, ps;
    float *turned, *across; // forward: the volume as [x][y][Wp], and as [y][x][Wp] (or null)
    float *lines;           // G or U as [kn][cols][Wp]
    Epilogue ep;
    int up;                 // backward: pixels per coarse pixel edge (refined detector), else 1
    int stage;              // backward: columns staged at a time
    int quads, rays;        // forward: lanes per ray (V of w each) and rays per wave
    int bx, by, parts, part_len;  // backward: bricks, angle parts
    float *partial;         // backward: the parts' sums ([entry][part][z][y][x]), null for one part
    int chunks;             // chunks of w
};

template <int N>
struct FlatArgs {
    FlatView v[N];
    int begin[N + 1];
    int n;
    int shift;  // chunk size of the XCD order (xcd_logical)
};

// Kernels take the arguments of one instance or of up to FLAT_MAX: those of a
// full launch are 3.5 KB, which cost small calls 0.5 us on the host and 3 us
// until their blocks had read them.
using FlatOne = FlatArgs<1>;
using FlatMulti = FlatArgs<FLAT_MAX>;

template <int ZL>
struct FlatVec {
    float v[ZL];
};


template <int ZL>
__device__ __forceinline__ FlatVec<ZL> flat_load(const float *p)
{
    FlatVec<ZL> r;
    if constexpr (ZL == 4) {
        const float4 t = *reinterpret_cast<const float4 *>(p);
        r.v[0] = t.x;
        r.v[1] = t.y;
        r.v[2] = t.z;
        r.v[3] = t.w;
    } else if constexpr (ZL == 2) {
        const float2 t = *reinterpret_cast<const float2 *>(p);
        r.v[0] = t.x;
        r.v[1] = t.y;
    } else {
        r.v[0] = *p;
    }
    return r;
}

template <int ZL>
__device__ __forceinline__ void flat_store(float *p, const FlatVec<ZL> &r)
{
    if constexpr (ZL == 4)
        *reinterpret_cast<float4 *>(p) = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
    else if constexpr (ZL == 2)
        *reinterpret_cast<float2 *>(p) = make_float2(r.v[0], r.v[1]);
    else
        *p = r.v[0];
}

__device__ __forceinline__ float lane_f(float v, int lane)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

__device__ __forceinline__ int lane_i(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// ---------------------------------------------------------------------------
// layout passes: 32 x 32 tiles through LDS, blocks of 32 x 8 threads
// ---------------------------------------------------------------------------

// turned[x][y][w], and across[y][x][w] where it is asked for, from vol[z][y][x]
// of every entry: a block per tile of 32 x by 32 w of one y.
__host__ __device__ inline int64_t flat_turn_blocks(const FlatView &v)
{
    return (int64_t)((v.nx + 31) / 32) * ((v.W + 31) / 32) * v.ny;
}

// The line of zeros after `lines` lines of pitch Wp (written by the blocks of
// a layout pass that start at w0, for the w of their tile).
__device__ __forceinline__ void flat_zero_line(float *base, int64_t lines, int Wp, int w0)
{
    const int w = w0 + threadIdx.x;
    if (threadIdx.y == 0 && w < Wp) base[lines * Wp + w] = 0.0f;
}

template <typename Args>
__global__ void __launch_bounds__(256) flat_turn(Args M)
{
    __shared__ float tile[32][33];
    const int k = owner_of(M.begin, (int)blockIdx.x);
    const FlatView &v = M.v[k];
    const int id = (int)blockIdx.x - M.begin[k];
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int tiles_x = (v.nx + 31) / 32, tiles_w = (v.W + 31) / 32;
    const int x0 = (id % tiles_x) * 32, y = (id / tiles_x) % v.ny, w0 = (id / (tiles_x * v.ny)) * 32;
    if (w0 >= tiles_w * 32) return;
    int b = (w0 + ty) / v.nz, z = w0 + ty - b * v.nz;
    for (int r = ty; r < 32; r += 8) {
        const int x = x0 + tx;
        float t = 0.0f;
        if (w0 + r < v.W && x < v.nx) t = v.vol[b * v.vs + ((int64_t)z * v.ny + y) * v.nx + x];
        tile[r][tx] = t;
        for (z += 8; z >= v.nz; z -= v.nz) ++b;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int x = x0 + r, w = w0 + tx;
        if (x < v.nx && w < v.Wp) {
            v.turned[((int64_t)x * v.ny + y) * v.Wp + w] = tile[tx][r];
            if (v.across) v.across[((int64_t)y * v.nx + x) * v.Wp + w] = tile[tx][r];
        }
    }
    if (x0 == 0 && y == 0) {
        flat_zero_line(v.turned, (int64_t)v.nx * v.ny, v.Wp, w0);
        if (v.across) flat_zero_line(v.across, (int64_t)v.nx * v.ny, v.Wp, w0);
    }
}

// y[i, a, j] = l lerp_t G[a, j, .] through the epilogue: a block per tile of
// 32 columns by 32 (entry, row) of one angle.
__host__ __device__ inline int64_t flat_rows_blocks(const FlatView &v)
{
    return (int64_t)((v.cols + 31) / 32) * ((v.W / v.nz * v.rows + 31) / 32) * v.kn;
}

// Interpolation of one detector row in a line: the value at z and the next
// one with weight w (z = -2: the row misses the volume).
struct FlatRow {
    int z;
    float w;
};

__device__ __forceinline__ FlatRow flat_row(const FlatAngle &A, int i, int j, int nz)
{
    const double t = A.t0 + (double)j * A.tj + (double)i * A.tv;
    FlatRow r = {-2, 0.0f};
    if (t > -1.0 && t < (double)nz) {
        const double f = floor(t);
        r.z = (int)f;
        r.w = (float)(t - f);
    }
    return r;
}

template <typename Args>
__global__ void __launch_bounds__(256) flat_rows(Args M)
{
    __shared__ float tile[32][33];
    __shared__ FlatRow rows_of[32];
    __shared__ int entry_of[32], index_of[32];
    const int q = owner_of(M.begin, (int)blockIdx.x);
    const FlatView &v = M.v[q];
    const int id = (int)blockIdx.x - M.begin[q];
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int tiles_j = (v.cols + 31) / 32, all = v.W / v.nz * v.rows;
    const int j0 = (id % tiles_j) * 32, k = (id / tiles_j) % v.kn, r0 = (id / (tiles_j * v.kn)) * 32;
    if (r0 >= all) return;
    const FlatAngle &A = v.ang[k];
    // (the row's place in a line is the same for every column unless the
    // detector's u axis leaves the slices: formed once per row then, as the
    // FP64 positions and divisions would otherwise bound this pass)
    const bool level = A.tj == 0.0;
    if (ty == 0) {
        const int b = (r0 + tx) / v.rows, i = r0 + tx - b * v.rows;
        entry_of[tx] = b;
        index_of[tx] = i;
        rows_of[tx] = flat_row(A, i, 0, v.nz);
    }
    __syncthreads();
    const int b = entry_of[tx], i = index_of[tx];
    const FlatRow fr = rows_of[tx];
    const float *g0 = v.lines + ((int64_t)k * v.cols + j0) * v.Wp + b * v.nz;
    for (int c = ty; c < 32; c += 8) {
        float y = 0.0f;
        if (j0 + c < v.cols && r0 + tx < all) {
            const FlatRow r = level ? fr : flat_row(A, i, j0 + c, v.nz);
            if (r.z > -2) {
                const float *g = g0 + (int64_t)c * v.Wp + r.z;
                const float lo = r.z >= 0 ? g[0] : 0.0f, hi = r.z + 1 < v.nz ? g[1] : 0.0f;
                y = A.len * fmaf(r.w, hi - lo, lo);
            }
        }
        tile[c][tx] = y;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8)
        if (r0 + r < all && j0 + tx < v.cols)
            emit(v.proj + entry_of[r] * v.ps, ((int64_t)index_of[r] * v.n_angles + A.a) * v.cols + j0 + tx, entry_of[r],
                 tile[tx][r], v.ep);
}

// U[a, j, z] = sum_i L(t - z) l y[i, a, j]: a block per tile of 32 columns by
// 32 w of one angle. The rows i with |t - z| < 1 are found in FP64 (t is
// affine in i), and read along the columns.
__host__ __device__ inline int64_t flat_splat_blocks(const FlatView &v)
{
    return (int64_t)((v.cols + 31) / 32) * ((v.W + 31) / 32) * v.kn;
}

// The detector rows i .. i + n - 1 with a weight at height z: row i + e has
// the weight 1 - |d + e tv| (FP64 position of the first, rows at most a few).
struct FlatSpan {
    int i, n;
    float d;
};

__device__ __forceinline__ FlatSpan flat_span(const FlatAngle &A, int z, int j, int rows)
{
    const double tt = A.t0 + (double)j * A.tj, inv = 1.0 / A.tv, half = fabs(inv), mid = ((double)z - tt) * inv;
    const int lo = (int)fmax(0.0, ceil(mid - half)), hi = (int)fmin((double)(rows - 1), floor(mid + half));
    FlatSpan s = {lo, max(0, hi - lo + 1), (float)(tt + (double)lo * A.tv - (double)z)};
    return s;
}

template <typename Args>
__global__ void __launch_bounds__(256) flat_splat(Args M)
{
    __shared__ float tile[32][33];
    __shared__ FlatSpan spans[32];
    __shared__ int entry_of[32];
    const int q = owner_of(M.begin, (int)blockIdx.x);
    const FlatView &v = M.v[q];
    const int id = (int)blockIdx.x - M.begin[q];
    const int tx = threadIdx.x, ty = threadIdx.y;
    const int tiles_j = (v.cols + 31) / 32;
    const int j0 = (id % tiles_j) * 32, k = (id / tiles_j) % v.kn, w0 = (id / (tiles_j * v.kn)) * 32;
    if (w0 >= v.W) return;
    const FlatAngle &A = v.ang[k];
    const bool level = A.tj == 0.0;  // (as in flat_rows)
    if (ty == 0) {
        entry_of[tx] = (w0 + tx) / v.nz;
        spans[tx] = flat_span(A, w0 + tx - entry_of[tx] * v.nz, 0, v.rows);
    }
    __syncthreads();
    const int j = j0 + tx, up = v.up, coarse = up == 1 ? v.cols : v.cols / up;
    const float scale = A.len / (float)(up * up), tv = (float)A.tv;
    const int64_t line = (int64_t)v.n_angles * coarse;
    const float *col = v.proj + (int64_t)A.a * coarse + (up == 1 ? j : j / up);
    for (int r = ty; r < 32; r += 8) {
        float u = 0.0f;
        if (j < v.cols && w0 + r < v.W) {
            const int b = entry_of[r];
            const FlatSpan s = level ? spans[r] : flat_span(A, w0 + r - b * v.nz, j, v.rows);
            const float *y = col + b * v.ps;
            for (int e = 0; e < s.n; ++e) {
                const float wgt = 1.0f - fabsf(fmaf((float)e, tv, s.d));
                // (rows of no weight are not read: they may hold infinities)
                if (wgt > 0.0f) u = fmaf(wgt, scale * y[(up == 1 ? s.i + e : (s.i + e) / up) * line], u);
            }
        }
        tile[r][tx] = u;
    }
    __syncthreads();
    for (int c = ty; c < 32; c += 8) {
        const int jc = j0 + c, w = w0 + tx;
        if (jc < v.cols && w < v.Wp) v.lines[((int64_t)k * v.cols + jc) * v.Wp + w] = tile[tx][c];
    }
}

// ---------------------------------------------------------------------------
// forward: G[a, j, w]
// ---------------------------------------------------------------------------
template <int V>
__device__ __forceinline__ FlatVec<V> flat_bload(__amdgpu_buffer_rsrc_t rs, uint32_t bytes)
{
    if constexpr (V == 4)
        return __builtin_bit_cast(FlatVec<4>, __builtin_amdgcn_raw_buffer_load_b128(rs, bytes, 0, 0));
    else if constexpr (V == 2)
        return __builtin_bit_cast(FlatVec<2>, __builtin_amdgcn_raw_buffer_load_b64(rs, bytes, 0, 0));
    else
        return __builtin_bit_cast(FlatVec<1>, __builtin_amdgcn_raw_buffer_load_b32(rs, bytes, 0, 0));
}

// A wave takes `rays` neighbouring detector columns of one angle and V quads
// of w (lane: ray lane / quads, V consecutive w at V (lane % quads); V = 1 and
// 2 on lines of one and two w). Slice by slice every ray takes the two voxel
// columns beside it straight from memory (the line of zeros after the last one
// where they lie beyond the volume). Where a ray has several lanes, the weights
// and addresses of up to 32 slices are formed by all lanes (FP64 positions) and
// passed on through LDS; where it has one (OWN), that lane forms its own.
// Slices are summed in groups of FLAT_SUM, whose sums are added in order.
//
// A block takes four neighbouring angles, whose rays meet nearly the same voxel
// columns, or one angle, whose groups its four waves take in turn (SPLIT: few
// rays, which would leave the chip waiting on one wave's loads per SIMD). The
// launch goes through chunks of at most 80 of w, in a chunk through strips of 8
// column tiles, in a strip through the angles: the blocks that an XCD runs
// together meet few voxel columns, so that its L2 holds them (512^3, 360
// angles: 9.9 ms; angles before tiles, chunks of 256 of w: 19.4 ms).
//
// Bound: the L1 port and L2 (two 16-byte loads per lane, 8 fma, one LDS read
// for 4 samples; its address unit 74 % busy at 8 x 128^3, 85 % at 75 x 441^2).
// fp_padded with its layouts against this with both layout passes, pixel pitch
// sqrt 2 (in brackets 1):
//   64^3, 180 angles      59 (66) and 30 (30) us
//   128^3, 360 angles    0.38 (0.52) and 0.16 (0.20) ms
//   256^3, 360 angles    2.06 (3.35) and 1.05 (1.36) ms
//   512^3, 360 angles    15.1 and 9.3 ms
//   75 x 441 x 441, 361  1.69 (2.73) and 1.16 (1.37) ms
//   16 x (256 x 256), 180 angles 123 (137) and 65 (73) us
//   1 x (256 x 256), 180 angles 60 (68) and 32 (31) us, 4 of them 65 (73) and 33 (37)
//   1 x (512 x 512), 360 angles 292 (371) and 134 (119) us
//   2 x (1024 x 1024), 720 angles 1.14 (1.33) and 0.69 (0.87) ms
// Taken back: lines staged in LDS by blocks that go through the slices in step
// (a barrier per slice: 200^3, 360 angles, pitch sqrt 2 1.07 ms against 0.72
// here; few blocks on small volumes: 80^3, 60 angles 0.09 against 0.03); one ray
// per wave with weights from readlane (1.15 ms).
template <int V, bool OWN, bool SPLIT, typename Args>
__global__ void __launch_bounds__(256) fp_flat(Args M)
{
    constexpr int UN = 8;  // slices whose columns are in flight together
    extern __shared__ __align__(16) float flat_lds[];
    const int logical = xcd_logical(M.shift);
    if (logical >= M.begin[M.n]) return;
    const int inst = owner_of(M.begin, logical);
    const FlatView &v = M.v[inst];
    const int id = logical - M.begin[inst];
    const int cols = v.cols, Wp = v.Wp, L = OWN ? 1 : v.quads, R = v.rays, NS = OWN ? UN : v.stage;
    const int tiles = (cols + R - 1) / R, ks = SPLIT ? v.kn : (v.kn + 3) / 4;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int T = FLAT_STRIP;
    const int per = ks * tiles, chunk = id / per, in_chunk = id - chunk * per;
    const int strip = in_chunk / (ks * T), width = min(T, tiles - strip * T), in_strip = in_chunk - strip * ks * T;
    const int jb = (strip * T + in_strip % width) * R, w0 = chunk * V * L;
    const int k = SPLIT ? in_strip / width : in_strip / width * 4 + wv;
    if (k >= v.kn) return;  // (never with SPLIT, whose waves meet at barriers)
    float4 *entry = reinterpret_cast<float4 *>(flat_lds) + wv * NS * R;
    typedef const __attribute__((address_space(4))) FlatAngle ConstAngle;
    ConstAngle &A = ((ConstAngle *)v.ang)[k];
    const int m = A.m;
    const int nm = m == 0 ? v.nx : v.ny, nc = m == 0 ? v.ny : v.nx;
    const bool turned = m == 0 || !v.across;
    // voxel column (n, c) is n sn + c sc
    const int sn = m == 0 ? v.ny : (turned ? 1 : v.nx), sc = m == 0 || !turned ? 1 : v.ny;
    const int nref = nm / 2, zero = v.nx * v.ny;
    // the ray of column j: q(n) = base + j qj + (n - nref) qm, slices with q in (-1, nc)
    const double base = fma(A.qm, (double)nref, A.q0);
    const auto ray_at = [&](int ray) {  // (held where the voxel columns' numbers are exact)
        return fmin(fmax(fma(A.qj, (double)min(jb + ray, cols - 1), base), -1e8), 1e8);
    };
    const double Rd = ray_at(lane % R);
    int lo = 0, hi = nm - 1;
    if (A.qm != 0.0) {
        const double t0 = (-1.0 - Rd) / A.qm, t1 = ((double)nc - Rd) / A.qm;
        lo = max(0, (int)fmin(fmax(ceil(fmin(t0, t1) + nref), -1e9), 1e9));
        hi = min(nm - 1, (int)fmax(fmin(floor(fmax(t0, t1) + nref), 1e9), -1e9));
    } else if (!(Rd > -1.0 && Rd < (double)nc)) {
        hi = -1;
    }
    if (lo > hi) {
        lo = nm;
        hi = -1;
    }
    lo = __builtin_amdgcn_readfirstlane(wave_min(lo));
    hi = __builtin_amdgcn_readfirstlane(wave_max(hi));
    const int r = lane / L, w = w0 + (lane - r * L) * V;
    const bool live = r < R && w < Wp;
    const uint32_t lane_bytes = (uint32_t)w * 4u, line_bytes = (uint32_t)Wp * 4u;
    const uint32_t n_bytes = (uint32_t)sn * line_bytes, c_bytes = (uint32_t)sc * line_bytes, none = (uint32_t)zero * line_bytes;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void *)(turned ? v.turned : v.across), (short)0,
                                          (int)((uint32_t)(zero + 1) * line_bytes), 0x00020000);
    // weight and addresses of the two voxel columns beside a ray in slice n (byte offset at)
    const bool narrow = c_bytes < 1u << 24 && nc < 1 << 24;
    const auto place = [&](double q, uint32_t at, bool inside, float &wh, uint32_t &ra, uint32_t &rb) {
        const double f = floor(q);
        const int c = (int)f;
        wh = (float)(q - f);
        rb = at + (narrow ? __umul24((uint32_t)(c + 1), c_bytes) : (uint32_t)(c + 1) * c_bytes);
        ra = inside && (unsigned)c < (unsigned)nc ? rb - c_bytes : none;
        rb = inside && (unsigned)(c + 1) < (unsigned)nc ? rb : none;
    };
    // acc += the slices of (1 - wh, wh, ra, rb)
    const auto sample = [&](const float4 (&t)[UN], FlatVec<V> &acc) {
        FlatVec<V> a[UN], b[UN];
#pragma unroll
        for (int e = 0; e < UN; ++e) {
            a[e] = flat_bload<V>(rs, __builtin_bit_cast(uint32_t, t[e].z) + lane_bytes);
            b[e] = flat_bload<V>(rs, __builtin_bit_cast(uint32_t, t[e].w) + lane_bytes);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < UN; ++e)
#pragma unroll
            for (int z = 0; z < V; ++z) acc.v[z] = fmaf(t[e].y, b[e].v[z], fmaf(t[e].x, a[e].v[z], acc.v[z]));
        __builtin_amdgcn_sched_barrier(0);
    };
    // (ray, slice) of the lane's first entry of a step, and the way from one to the next
    const int h0 = lane / R, ray0 = lane - h0 * R, step_h = 64 / R, step_r = 64 - step_h * R;
    // the sum over the slices of one group of FLAT_SUM
    const auto group = [&](int g, FlatVec<V> &acc) {
#pragma unroll
        for (int z = 0; z < V; ++z) acc.v[z] = 0.0f;
        const int end = min(hi, g * FLAT_SUM + FLAT_SUM - 1);
        for (int n0 = max(g * FLAT_SUM, lo / NS * NS); n0 <= end; n0 += NS) {
            if constexpr (OWN) {
                if (!live) continue;
                const double dn = (double)(n0 - nref);
                float4 t[UN];
#pragma unroll
                for (int e = 0; e < UN; ++e) {
                    float wh;
                    uint32_t ra, rb;
                    place(fma(dn + (double)e, A.qm, Rd), (uint32_t)(n0 + e) * n_bytes, n0 + e <= end, wh, ra, rb);
                    t[e] = make_float4(1.0f - wh, wh, __builtin_bit_cast(float, ra), __builtin_bit_cast(float, rb));
                }
                sample(t, acc);
            } else {
                int h = h0, ray = ray0;
                for (int e = lane; e < NS * R; e += 64) {
                    const int n = n0 + h;
                    float wh;
                    uint32_t ra, rb;
                    place(fma((double)(n - nref), A.qm, step_r ? ray_at(ray) : Rd), (uint32_t)n * n_bytes, n <= end, wh, ra, rb);
                    entry[e] = make_float4(1.0f - wh, wh, __builtin_bit_cast(float, ra), __builtin_bit_cast(float, rb));
                    ray += step_r;
                    h += step_h;
                    if (ray >= R) {
                        ray -= R;
                        ++h;
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (live) {
                    const float4 *in = entry + r;
                    for (int h = 0; h < NS && n0 + h <= end; h += UN) {
                        float4 t[UN];
#pragma unroll
                        for (int e = 0; e < UN; ++e) t[e] = in[(h + e) * R];
                        sample(t, acc);
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
    };
    FlatVec<V> sum;  // of the groups, in their order
#pragma unroll
    for (int z = 0; z < V; ++z) sum.v[z] = 0.0f;
    const int last = hi / FLAT_SUM;
    if constexpr (SPLIT) {
        // a group per wave; their sums are added in order by the first wave
        FlatVec<V> *part = reinterpret_cast<FlatVec<V> *>(flat_lds + (OWN ? 0 : 4 * 4 * NS * R));
        int buf = 0;
        for (int g = lo / FLAT_SUM; lo <= hi && g <= last; g += 4, buf ^= 1) {
            FlatVec<V> acc;
            group(g + wv, acc);  // (past the last one: nothing)
            part[(buf * 4 + wv) * 64 + lane] = acc;
            __syncthreads();
            if (wv == 0)
                for (int s = 0; s < 4 && g + s <= last; ++s)
#pragma unroll
                    for (int z = 0; z < V; ++z) sum.v[z] += part[(buf * 4 + s) * 64 + lane].v[z];
        }
        if (wv != 0) return;
    } else {
        for (int g = lo / FLAT_SUM; lo <= hi && g <= last; ++g) {
            FlatVec<V> acc;
            group(g, acc);
#pragma unroll
            for (int z = 0; z < V; ++z) sum.v[z] += acc.v[z];
        }
    }
    if (live && jb + r < cols) flat_store<V>(v.lines + ((int64_t)k * cols + jb + r) * Wp + w, sum);
}

// ---------------------------------------------------------------------------
// backward: x[n, c, w] from U
// ---------------------------------------------------------------------------
// Four neighbouring values of one output row through the epilogue (as emit).
__device__ __forceinline__ void emit4(float *out, int64_t o, int64_t b, float4 a, const Epilogue &e)
{
    float4 *p = reinterpret_cast<float4 *>(out + o);
    if (e.mode == EP_SET) {
        *p = a;
        return;
    }
    float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (e.mode != EP_RESIDUAL) r = *p;
    if (e.mode == EP_ADD) {
        *p = make_float4(r.x + a.x, r.y + a.y, r.z + a.z, r.w + a.w);
        return;
    }
    const int64_t q = b * e.stride + o;
    const float4 w = *reinterpret_cast<const float4 *>(e.w + q);
    if (e.mode == EP_RESIDUAL) {
        const float4 y = *reinterpret_cast<const float4 *>(e.y + q);
        r = make_float4(w.x * (y.x - a.x), w.y * (y.y - a.y), w.z * (y.z - a.z), w.w * (y.w - a.w));
    } else if (e.mode == EP_SCALED_ADD) {
        r = make_float4(r.x + w.x * a.x, r.y + w.y * a.y, r.z + w.z * a.z, r.w + w.w * a.w);
    } else {
        r = make_float4(r.x - w.x * a.x, r.y - w.y * a.y, r.z - w.z * a.z, r.w - w.w * a.w);
    }
    *p = r;
}

// Whether an instance's output rows (or voxels, where `row` is their number)
// and its epilogue's data can be taken four at a time.
__host__ __device__ __forceinline__ bool flat_quads(const FlatView &v, int64_t row)
{
    return (row & 3) == 0 && (((uintptr_t)v.vol | (uintptr_t)v.ep.y | (uintptr_t)v.ep.w) & 15) == 0 &&
           ((v.vs | v.ep.stride) & 3) == 0;
}

// Writes a wave's 16 neighbouring voxel columns (x0 .., y), ZL of w per lane from
// w0 on. Where four voxels of a row can be written at once, a lane writes its own;
// else the sums go through a tile of the wave's own in LDS, so that 16 lanes write
// neighbouring voxels: a voxel at a time from each lane, every store met 64 cache
// lines, which cost more than the sums of few angles (8 angles: 150^3 48 us, 32 us
// through the tile; 200 x 150^2 42 and 32 us).
constexpr int FLAT_TILE = 64 * (FLAT_BX + 1);  // floats of a wave's tile

template <int ZL>
__device__ __forceinline__ void flat_write(const FlatView &v, int part, int x0, int y, int w0,
                                           const FlatVec<ZL> (&acc)[FLAT_BX], float *tile)
{
    static_assert(FLAT_BX == 16, "four rows of 16 voxels per store");
    const int lane = threadIdx.x & 63;
    const int64_t ve = (int64_t)v.nx * v.ny * v.nz;
    Epilogue ep = v.ep;
    if (v.partial) ep.mode = EP_SET;
    const auto volume = [&](int b) { return v.partial ? v.partial + ((int64_t)b * v.parts + part) * ve : v.vol + b * v.vs; };
    if (flat_quads(v, v.nx)) {
        if (y >= v.ny) return;
#pragma unroll
        for (int z = 0; z < ZL; ++z) {
            const int w = w0 + lane * ZL + z;
            if (w >= v.W) continue;
            const int b = w / v.nz, iz = w - b * v.nz;
            const int64_t o = ((int64_t)iz * v.ny + y) * v.nx + x0;
#pragma unroll
            for (int c = 0; c < FLAT_BX; c += 4)
                if (x0 + c < v.nx)
                    emit4(volume(b), o + c, b,
                          make_float4(acc[c].v[z], acc[c + 1].v[z], acc[c + 2].v[z], acc[c + 3].v[z]), ep);
        }
        return;
    }
    __syncthreads();  // (the tile lies where the block staged its lines)
    if (y >= v.ny) return;
    const int col = lane % FLAT_BX, first = lane / FLAT_BX;
    constexpr int STEP = 64 / FLAT_BX * ZL;  // in w, from one store to the next
#pragma unroll
    for (int z = 0; z < ZL; ++z) {
        wave_lds_sync();
#pragma unroll
        for (int c = 0; c < FLAT_BX; ++c) tile[lane * (FLAT_BX + 1) + c] = acc[c].v[z];
        wave_lds_sync();
        int w = w0 + first * ZL + z, b = w / v.nz, iz = w - b * v.nz;
        for (int r = first; r < 64; r += 64 / FLAT_BX) {
            if (x0 + col < v.nx && w < v.W)
                emit(volume(b), ((int64_t)iz * v.ny + y) * v.nx + x0 + col, b, tile[r * (FLAT_BX + 1) + col], ep);
            w += STEP;
            iz += STEP;
            if (iz >= v.nz) {
                const int more = v.nz >= STEP ? 1 : iz / v.nz;
                b += more;
                iz -= more * v.nz;
            }
        }
    }
}

// Detector column of the ray through the voxel column (x, y); the first one
// with a weight there; and the weight of the e-th from it on, max(0, 1 - |j -
// jc| b2), from FP64 positions.
__device__ __forceinline__ double flat_column(const FlatAngle &A, double x, double y)
{
    return A.m == 0 ? fma(A.gc, y, fma(A.gm, x, A.g0)) : fma(A.gc, x, fma(A.gm, y, A.g0));
}

template <int NC>
__device__ __forceinline__ double flat_first(const FlatAngle &A, double jc)
{
    return fmin(fmax(NC == 2 ? floor(jc) : ceil(jc - fabs(A.gc)), -1e8), 1e8);
}

__device__ __forceinline__ float flat_weight(const FlatAngle &A, double j0, double jc, int e)
{
    return fmaxf(fmaf(-fabsf((float)(j0 - jc) + (float)e), A.b2, 1.0f), 0.0f);
}

// A block of 8 waves takes a brick of 16 x 8 voxel columns and 64 ZL of w, a
// wave the 16 columns of one y. Per angle the lines U of the detector columns
// that meet the brick are staged in LDS (two buffers, one barrier per angle),
// and every voxel column takes its NC detector columns (|j - jc| < 1 / b2 for
// b2 = |dq / dj|: two where a detector column is at least a voxel wide, as
// many as fit otherwise) with their weights, formed by the 64 lanes for four
// angles at once. A column without weight is taken from a staged line of
// zeros, so that an infinite or NaN pixel reaches no voxel that its ray does
// not meet.
//
// Bound: vector ALU and LDS together, in step with the barriers (0.6 vector
// instructions and 0.09 to 0.12 LDS reads of 8 to 16 bytes per lane and
// CU-cycle); per (voxel column, angle) NC + 1 readlane, NC addresses, NC reads
// and NC ZL fma (bp_wave: about 37 instructions per 64 voxels at pixel pitch 1,
// where its 16-voxel bricks take two chunks of columns). Two angles per step at
// ZL = 2 cost a block per CU (registers): 2.4 against 2.2 ms at 75 x 441 x 441,
// 361 angles, 75 x 623 (bp_wave: 5.8); 16 x 16 bricks 3.1. 8 x 128^3, 180
// angles, 128 x 192: 0.64 ms with the splat against 3.04.
template <int ZL, int NC, typename Args>
__global__ void __launch_bounds__(64 * FLAT_BY) bp_flat(Args M)
{
    extern __shared__ __align__(16) float flat_lds[];
    constexpr int CF = 64 * ZL, AL = 4;  // floats per staged column; angles whose weights a wave holds
    constexpr int SW = 3;  // columns staged by a wave in one pass
    const int logical = xcd_logical(M.shift);
    if (logical >= M.begin[M.n]) return;
    const int inst = owner_of(M.begin, logical);
    const FlatView &v = M.v[inst];
    int id = logical - M.begin[inst];
    const int bx = id % v.bx;
    id /= v.bx;
    const int by = id % v.by;
    id /= v.by;
    const int w0 = (id % v.chunks) * CF, part = id / v.chunks;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x0 = bx * FLAT_BX, y0 = by * FLAT_BY, kn = v.kn, cols = v.cols, Wp = v.Wp;
    const int ka = part * v.part_len, kb = min(kn, ka + v.part_len);
    const int w = w0 + lane * ZL;
    const int SC = v.stage;
    const FlatAngle *ang = v.ang;
    FlatVec<ZL> acc[FLAT_BX], next[SW];
#pragma unroll
    for (int c = 0; c < FLAT_BX; ++c)
#pragma unroll
        for (int z = 0; z < ZL; ++z) acc[c].v[z] = 0.0f;
    if (wv < 2) {  // the last place of each buffer: a line of zeros
        FlatVec<ZL> zero;
#pragma unroll
        for (int z = 0; z < ZL; ++z) zero.v[z] = 0.0f;
        flat_store<ZL>(flat_lds + (wv * (SC + 1) + SC) * CF + lane * ZL, zero);
    }
    // first staged detector column of angle ka + 64 i + lane
    int jbv = 0;
    auto bases = [&](int k) {
        const FlatAngle &A = ang[min(k + lane, kn - 1)];
        const double gx = A.m == 0 ? A.gm : A.gc, gy = A.m == 0 ? A.gc : A.gm;
        const double j = flat_column(A, x0, y0) + fmin(0.0, (FLAT_BX - 1) * gx) + fmin(0.0, (FLAT_BY - 1) * gy);
        jbv = (int)flat_first<NC>(A, j - 1e-6);
    };
    // (lanes past the last w read the line's last values; nothing of theirs is written)
    const float *src = v.lines + min(w, Wp - ZL);
    const int64_t line = Wp, line_by = (int64_t)Wp * FLAT_BY;
    // staged columns of pass e0 (SW columns of every wave) of angle k
    auto load = [&](int k, int e0) {
        const int j0 = lane_i(jbv, (k - ka) & 63) + wv + e0 * SW * FLAT_BY;
        const float *p = src + ((int64_t)k * cols + j0) * line;
#pragma unroll
        for (int e = 0; e < SW; ++e) {
            if ((unsigned)(j0 + e * FLAT_BY) < (unsigned)cols) {
                next[e] = flat_load<ZL>(p + e * line_by);
            } else {
#pragma unroll
                for (int z = 0; z < ZL; ++z) next[e].v[z] = 0.0f;
            }
        }
    };
    auto store = [&](float *buf, int e0) {
#pragma unroll
        for (int e = 0; e < SW; ++e) {
            const int s = wv + (e0 * SW + e) * FLAT_BY;
            if (s < SC) flat_store<ZL>(buf + s * CF, next[e]);
        }
    };
    bases(ka);
    load(ka, 0);
    int places = 0;  // lane (angle k % AL, column c): staged places of the voxel's detector columns, 8 bits each
    float wt[NC];
#pragma unroll
    for (int e = 0; e < NC; ++e) wt[e] = 0.0f;
    for (int k = ka; k < kb; ++k) {
        const int at = k - ka;
        if ((at & (AL - 1)) == 0) {
            const int jb = __shfl(jbv, (at & 63) + lane / FLAT_BX, 64);
            const FlatAngle &A = ang[min(k + lane / FLAT_BX, kn - 1)];
            const double jc = flat_column(A, x0 + lane % FLAT_BX, y0 + wv), j0 = flat_first<NC>(A, jc);
            const int first = min(max((int)j0 - jb, 0), SC - NC);
            places = 0;
#pragma unroll
            for (int e = 0; e < NC; ++e) {
                wt[e] = flat_weight(A, j0, jc, e);
                places |= (wt[e] > 0.0f ? first + e : SC) << (8 * e);
            }
        }
        float *buf = flat_lds + (at & 1) * (SC + 1) * CF + lane * ZL;
        store(buf, 0);
        for (int e0 = 1; e0 * SW * FLAT_BY < SC; ++e0) {  // (windows wider than one pass)
            load(k, e0);
            store(buf, e0);
        }
        __syncthreads();
        if (k + 1 < kb) {
            if (((at + 1) & 63) == 0) bases(k + 1);
            load(k + 1, 0);
        }
        constexpr int CB = ZL == 4 ? 2 : 4;  // voxel columns whose lines are in flight together
#pragma unroll
        for (int c0 = 0; c0 < FLAT_BX; c0 += CB) {
            FlatVec<ZL> u[CB][NC];
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                const uint32_t at4 = (uint32_t)lane_i(places, (at & (AL - 1)) * FLAT_BX + c0 + c);
#pragma unroll
                for (int e = 0; e < NC; ++e) u[c][e] = flat_load<ZL>(buf + ((at4 >> (8 * e)) & 255u) * CF);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int e = 0; e < NC; ++e) {
                    const float f = lane_f(wt[e], (at & (AL - 1)) * FLAT_BX + c0 + c);
#pragma unroll
                    for (int z = 0; z < ZL; ++z) acc[c0 + c].v[z] = fmaf(f, u[c][e].v[z], acc[c0 + c].v[z]);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    flat_write<ZL>(v, part, x0, y0 + wv, w0, acc, flat_lds + wv * FLAT_TILE);
}

// The same without staging, for short lines: a wave takes `rays` voxel columns
// and `quads` lanes of V consecutive w for each, so that lines of any length
// fill its lanes (one w per lane over 64 of them left 63 of 64 idle on a single
// slice), a block four waves' columns in a tile. The weights
// and places of up to 32 angles are formed by all lanes, a (column, angle) per
// lane, and passed on through LDS; columns of no weight are read past the end
// of the buffer, which gives zeros, so that an infinite pixel reaches no voxel
// that its ray does not meet. The angle parts run in blocks of their own, or in
// turn with their sums in registers (multiples of FLAT_PART angles).
//
// Bound: the L1 port (two 16-byte loads of 16 cycles each per 64 lanes; its
// address unit 81 % busy at 64 x 256^2, 66 % at 16). Whole backprojection, 180
// angles, pixel pitch 1, in brackets one w per lane and bp_wave: 256^2 42 us (250,
// 183), 16 slices of it 74 (260, 265), 64 209 (290, 1141).
// Columns along x of a block's tile of 4 rays (any shape takes the same time).
__host__ __device__ inline int flat_tile(int rays) { return rays % 4 == 0 ? 16 : (rays % 2 == 0 ? 8 : 4); }

constexpr int FLAT_PART = 4;

template <int V, int NC, typename Args>
__global__ void __launch_bounds__(256) bp_flat_short(Args M)
{
    constexpr int EN = NC == 2 ? 512 : 256;  // (angle, column) entries of a wave at a time
    constexpr int UN = NC == 2 ? 8 : 4;  // angles whose lines are in flight together
    constexpr int PART = FLAT_PART;
    constexpr uint32_t NONE = 0x80000000u;
    struct Entry {
        float w[NC];
        uint32_t at[NC];
    };
    __shared__ __align__(16) Entry entry[4][EN];
    const int logical = xcd_logical(M.shift);
    if (logical >= M.begin[M.n]) return;
    const int inst = owner_of(M.begin, logical);
    const FlatView &v = M.v[inst];
    int id = logical - M.begin[inst];
    const int bx = id % v.bx;
    id /= v.bx;
    const int by = id % v.by;
    id /= v.by;
    const int L = v.quads, R = v.rays, TX = flat_tile(R), rows = 4 * R / TX, cols = v.cols, Wp = v.Wp;
    const int w0 = (id % v.chunks) * V * L, part = id / v.chunks;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // (a block per angle part, or all parts in turn)
    const int ka = v.partial ? part * v.part_len : 0, kb = v.partial ? min(v.kn, ka + v.part_len) : v.kn;
    const int r = lane / L, w = w0 + (lane - r * L) * V;
    const int t0 = wv * R;  // the wave's first column of the tile
    const int x = bx * TX + (t0 + r) % TX, y = by * rows + (t0 + r) / TX;
    const bool live = r < R && w < Wp;
    const uint32_t lane_bytes = (uint32_t)w * 4u, line_bytes = (uint32_t)Wp * 4u, angle_bytes = (uint32_t)cols * line_bytes;
    // angles whose entries are formed together; (angle, column) of the lane's first one, and the way to the next
    const int NS = min(32, EN / R) / UN * UN;
    const int h0 = lane / R, c0 = lane - h0 * R, step_h = 64 / R, step_c = 64 - step_h * R;
    FlatVec<V> acc, sum;  // of the present part, of those before it
#pragma unroll
    for (int z = 0; z < V; ++z) acc.v[z] = sum.v[z] = 0.0f;
    int left = v.part_len;  // angles of the present part (a multiple of PART where several run in turn)
    for (int k0 = ka; k0 < kb; k0 += NS) {
        const int n = min(NS, kb - k0);
        int h = h0, c = c0;
        for (int e = lane; e < (n + UN - 1) / UN * UN * R; e += 64) {
            Entry t;
            const FlatAngle &A = v.ang[min(k0 + h, kb - 1)];
            const double jc = flat_column(A, bx * TX + (t0 + c) % TX, by * rows + (t0 + c) / TX);
            const double j0 = flat_first<NC>(A, jc);
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int j = (int)j0 + i;
                const float f = flat_weight(A, j0, jc, i);
                const bool some = h < n && f > 0.0f && (unsigned)j < (unsigned)cols;
                t.w[i] = some ? f : 0.0f;
                t.at[i] = some ? (uint32_t)h * angle_bytes + (uint32_t)j * line_bytes : NONE;
            }
            entry[wv][e] = t;
            c += step_c;
            h += step_h;
            if (c >= R) {
                c -= R;
                ++h;
            }
        }
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(v.lines + (int64_t)k0 * cols * Wp), (short)0, (int)((uint32_t)n * angle_bytes), 0x00020000);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (live) {
            const Entry *in = entry[wv] + r;
            for (int h = 0; h < n; h += UN) {
                Entry t[UN];
                FlatVec<V> u[UN][NC];
#pragma unroll
                for (int e = 0; e < UN; ++e) t[e] = in[(h + e) * R];
#pragma unroll
                for (int e = 0; e < UN; ++e)
#pragma unroll
                    for (int i = 0; i < NC; ++i) u[e][i] = flat_bload<V>(rs, t[e].at[i] + lane_bytes);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < UN; ++e) {
#pragma unroll
                    for (int i = 0; i < NC; ++i)
#pragma unroll
                        for (int z = 0; z < V; ++z) acc.v[z] = fmaf(t[e].w[i], u[e][i].v[z], acc.v[z]);
                    if (e % PART != PART - 1) continue;
                    left -= PART;
                    if (left == 0) {
                        left = v.part_len;
#pragma unroll
                        for (int z = 0; z < V; ++z) {
                            sum.v[z] += acc.v[z];
                            acc.v[z] = 0.0f;
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int z = 0; z < V; ++z) acc.v[z] = sum.v[z] + acc.v[z];
    if (!live || x >= v.nx || y >= v.ny) return;
#pragma unroll
    for (int z = 0; z < V; ++z) {
        if (w + z >= v.W) break;
        const int b = (w + z) / v.nz, iz = (w + z) - b * v.nz;
        const int64_t o = ((int64_t)iz * v.ny + y) * v.nx + x;
        if (v.partial)
            v.partial[((int64_t)b * v.parts + part) * ((int64_t)v.nx * v.ny * v.nz) + o] = acc.v[z];
        else
            emit(v.vol + b * v.vs, o, b, acc.v[z], v.ep);
    }
}

// The sums of the angle parts added in order and written through the
// epilogue: grid (voxels of the largest instance / 256 M.shift, entries,
// instances), M.shift voxels per thread: four where every instance allows it
// (flat_reduce_quads), or one. Bound: memory; 8 x 128^3, four parts: 94 us with
// one voxel per thread, 62 with four.
__host__ __device__ __forceinline__ bool flat_reduce_quads(const FlatView &v)
{
    return !v.partial || (flat_quads(v, (int64_t)v.nx * v.ny * v.nz) && ((uintptr_t)v.partial & 15) == 0);
}

template <typename Args>
__global__ void __launch_bounds__(256) flat_parts_reduce(Args M)
{
    const FlatView &v = M.v[blockIdx.z];
    const int64_t ve = (int64_t)v.nx * v.ny * v.nz, o = ((int64_t)blockIdx.x * 256 + threadIdx.x) * M.shift;
    const int b = blockIdx.y;
    if (!v.partial || o >= ve || b >= v.W / v.nz) return;
    const float *pp = v.partial + (int64_t)b * v.parts * ve + o;
    float *out = v.vol + b * v.vs;
    if (M.shift == 4) {
        FlatVec<4> t = flat_load<4>(pp);
#pragma unroll 4
        for (int s = 1; s < v.parts; ++s) {
            const FlatVec<4> u = flat_load<4>(pp + (int64_t)s * ve);
#pragma unroll
            for (int e = 0; e < 4; ++e) t.v[e] += u.v[e];
        }
        emit4(out, o, b, make_float4(t.v[0], t.v[1], t.v[2], t.v[3]), v.ep);
        return;
    }
    float t = pp[0];
    for (int s = 1; s < v.parts; ++s) t += pp[(int64_t)s * ve];
    emit(out, o, b, t, v.ep);
}

template <typename Args>
using FlatKernel = void (*)(Args);

template <typename A>
FlatKernel<A> fp_flat_kernel(int v, bool own, bool split)
{
    if (!own) return split ? fp_flat<4, false, true, A> : fp_flat<4, false, false, A>;
    if (v == 4) return split ? fp_flat<4, true, true, A> : fp_flat<4, true, false, A>;
    if (v == 2) return split ? fp_flat<2, true, true, A> : fp_flat<2, true, false, A>;
    return split ? fp_flat<1, true, true, A> : fp_flat<1, true, false, A>;
}

template <typename A>
FlatKernel<A> bp_flat_kernel(int zl, int nc)
{
    if (zl == 4) return nc == 2 ? bp_flat<4, 2, A> : (nc == 3 ? bp_flat<4, 3, A> : bp_flat<4, 4, A>);
    return nc == 2 ? bp_flat<2, 2, A> : (nc == 3 ? bp_flat<2, 3, A> : bp_flat<2, 4, A>);
}

template <typename A>
FlatKernel<A> bp_flat_short_kernel(int v, int nc)
{
    if (v == 4) return nc == 2 ? bp_flat_short<4, 2, A> : (nc == 3 ? bp_flat_short<4, 3, A> : bp_flat_short<4, 4, A>);
    return nc == 2 ? bp_flat_short<1, 2, A> : (nc == 3 ? bp_flat_short<1, 3, A> : bp_flat_short<1, 4, A>);
}

}  // namespace tsx
