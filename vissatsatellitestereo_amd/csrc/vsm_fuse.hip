// vsm_fuse.hip -- 2.5D DSM fusion kernels (HBM-bound, gfx950).
//
// Per view (reference aggregate_2p5d_util.py:45-106, lib/proj_to_grid.py:41-81,
// produce_dsm.py:46-58):
//   back-projection X = inv(P4) (col, row, 1, d), divide by X3, in FP64 with a
//   fixed operation order (compiled -ffp-contract=off) so grid indices are
//   bit-exact with the CPU restatement; row = floor((ul_n - N)/e_res),
//   col = floor((E - ul_e)/n_res) (the reference's xresolution/yresolution
//   pairing, lib/proj_to_grid.py:42-43); per-cell nanmax through a 64-bit
//   atomicMax on an order-preserving encoding of the FP64 height (max is
//   order-independent, so the raster does not depend on atomic ordering);
//   NaN cells filled with the median of the in-bounds non-NaN 3x3 neighbours
//   of the unfilled raster (lib/proj_to_grid.py:64-79), cast to float32;
//   3x3 median with replicated border (produce_dsm.py:58).
// Across views (aggregate_2p5d.py:66-81): cells with fewer than
// min_measurements values -> NaN, median, MAD = median |x - med|, drop
// |x - med| > MAD, mean (FP64 accumulation), then the 3x3 median.
// Median rule (NaN-aware): NaN excluded; even count -> mean of the two middle
// values; no values -> NaN.
#include "vsm_device.h"
#include "vsm_geo.h"
#include "vsm_kernels.h"

#include <algorithm>
#include <mutex>
#include <vector>

namespace vsm {

__device__ __forceinline__ unsigned long long enc_f64(double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b & 0x8000000000000000ull) ? ~b : (b | 0x8000000000000000ull);
}
__device__ __forceinline__ double dec_f64(unsigned long long k)
{
    const unsigned long long b = (k & 0x8000000000000000ull) ? (k & 0x7FFFFFFFFFFFFFFFull) : ~k;
    return __longlong_as_double((long long)b);
}

__device__ __forceinline__ void cell_of(const DsmGridDev &g, double E, double N, int &row, int &col,
                                        bool &ok)
{
    const double fr = floor((g.ul_n - N) / g.e_res);
    const double fc = floor((E - g.ul_e) / g.n_res);
    ok = fr >= 0.0 && fc >= 0.0 && fr < (double)g.n_size && fc < (double)g.e_size;
    row = ok ? (int)fr : 0;
    col = ok ? (int)fc : 0;
}

// One thread per depth pixel; d <= 0 or non-finite -> no point
// (aggregate_2p5d_util.py:76, 92-93).  GEO: the ENU point goes through
// local_to_global + latlon_to_eastnorh (aggregate_2p5d_util.py:95-98) and the
// cell value is the altitude.
template <bool GEO>
__global__ __launch_bounds__(256) void k_rasterize_view(const float *__restrict__ depth, int W, int H,
                                 const double *__restrict__ Mi, DsmGridDev g, vsm_geo_frame gf,
                                 unsigned long long *__restrict__ cell_max)
{
    // 64 x 4 pixels a workgroup: rows and columns without a division
    const int px = blockIdx.x * 64 + (threadIdx.x & 63), py = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (px >= W || py >= H) return;
    const float d32 = depth[(size_t)py * W + px];
    if (!(d32 > 0.f) || !isfinite(d32)) return;
    const double col = (double)px, row = (double)py, d = (double)d32;
    double X[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        X[i] = ((Mi[4 * i + 0] * col + Mi[4 * i + 1] * row) + Mi[4 * i + 2]) + Mi[4 * i + 3] * d;
    double E = X[0] / X[3], N = X[1] / X[3], h = X[2] / X[3];
    if (!isfinite(E) || !isfinite(N) || !isfinite(h)) return;
    if (GEO) {
        double Eu, Nu, alt;
        if (!geo::enu_to_utm(gf, E, N, h, Eu, Nu, alt)) return;
        E = Eu;
        N = Nu;
        h = alt;
    }
    int r, c;
    bool ok;
    cell_of(g, E, N, r, c, ok);
    if (!ok) return;
    atomicMax(&cell_max[(size_t)r * g.e_size + c], enc_f64(h));
}

__global__ void k_rasterize_points(const double *__restrict__ pts, long long n, DsmGridDev g,
                                   unsigned long long *__restrict__ cell_max)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double E = pts[3 * i], N = pts[3 * i + 1], h = pts[3 * i + 2];
    if (isnan(h) || isnan(E) || isnan(N)) return;
    int r, c;
    bool ok;
    cell_of(g, E, N, r, c, ok);
    if (!ok) return;
    atomicMax(&cell_max[(size_t)r * g.e_size + c], enc_f64(h));
}

__global__ void k_enu_to_utm(const double *__restrict__ enu, long long n, vsm_geo_frame gf,
                             double *__restrict__ out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double E, N, alt;
    const bool ok = geo::enu_to_utm(gf, enu[3 * i], enu[3 * i + 1], enu[3 * i + 2], E, N, alt);
    const double nan = __longlong_as_double(0x7FF8000000000000ll);
    out[3 * i] = ok ? E : nan;
    out[3 * i + 1] = ok ? N : nan;
    out[3 * i + 2] = ok ? alt : nan;
}

// ---------------------------------------------------------------------------
// 3D fusion: one thread per pixel of image i (see vsm_fuse_points).  FP64
// projections with a fixed operation order, FP32 normals.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void backproject4(const double *Mi, double col, double row, double d,
                                             double &X, double &Y, double &Z)
{
    double h[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        h[k] = ((Mi[4 * k + 0] * col + Mi[4 * k + 1] * row) + Mi[4 * k + 2]) + Mi[4 * k + 3] * d;
    X = h[0] / h[3];
    Y = h[1] / h[3];
    Z = h[2] / h[3];
}

__device__ __forceinline__ void project3(const double *P, double X, double Y, double Z, double &u0,
                                         double &u1, double &u2)
{
    u0 = ((P[0] * X + P[1] * Y) + P[2] * Z) + P[3];
    u1 = ((P[4] * X + P[5] * Y) + P[6] * Z) + P[7];
    u2 = ((P[8] * X + P[9] * Y) + P[10] * Z) + P[11];
}

__device__ __forceinline__ void rotate_normal(const float *R, const float *n, float &a, float &b,
                                              float &c)
{
    a = (R[0] * n[0] + R[1] * n[1]) + R[2] * n[2];
    b = (R[3] * n[0] + R[4] * n[1]) + R[5] * n[2];
    c = (R[6] * n[0] + R[7] * n[1]) + R[8] * n[2];
}

// Fuses pixel p of image i; true where it makes a point.
__device__ __forceinline__ bool fuse_pixel(const Fuse3dView *__restrict__ V, int i, const Fuse3dConst &k,
                                           long long p, FusedPoint &o)
{
    const Fuse3dView &A = V[i];
    const float d = A.depth[p];
    if (!(d > 0.f) || !isfinite(d)) return false;
    const double col = (double)(p % A.W), row = (double)(p / A.W);
    double X, Y, Z;
    backproject4(A.Pinv, col, row, (double)d, X, Y, Z);
    if (!isfinite(X) || !isfinite(Y) || !isfinite(Z)) return false;
    float na, nb, nc;
    rotate_normal(A.R, A.normal + 3 * p, na, nb, nc);
    int count = 1;
    double sx = X, sy = Y, sz = Z;
    float snx = na, sny = nb, snz = nc;
    uint32_t sg = A.gray ? A.gray[p] : 0u;
    for (int j = 0; j < k.n; ++j) {
        if (j == i) continue;
        const Fuse3dView &B = V[j];
        double u0, u1, u2;
        project3(B.P, X, Y, Z, u0, u1, u2);
        if (!(u2 > 0.0)) continue;
        const double cx = floor(u0 / u2 + 0.5), cy = floor(u1 / u2 + 0.5);
        if (!(cx >= 0.0 && cy >= 0.0 && cx < (double)B.W && cy < (double)B.H)) continue;
        const long long q = (long long)cy * B.W + (long long)cx;
        const float dj = B.depth[q];
        if (!(dj > 0.f) || !isfinite(dj)) continue;
        double Xj, Yj, Zj;
        backproject4(B.Pinv, cx, cy, (double)dj, Xj, Yj, Zj);
        const double ex = Xj - X, ey = Yj - Y, ez = Zj - Z;
        if (!(sqrt((ex * ex + ey * ey) + ez * ez) <= k.max_depth_err)) continue;
        double v0, v1, v2;
        project3(A.P, Xj, Yj, Zj, v0, v1, v2);
        if (!(v2 > 0.0)) continue;
        const double rx = v0 / v2 - col, ry = v1 / v2 - row;
        if (!(sqrt(rx * rx + ry * ry) <= k.max_reproj)) continue;
        float ma, mb, mc;
        rotate_normal(B.R, B.normal + 3 * q, ma, mb, mc);
        if (!((na * ma + nb * mb) + nc * mc >= k.cos_max_normal)) continue;
        if (j < i) return false;           // the cluster belongs to image j
        ++count;
        sx = sx + Xj;
        sy = sy + Yj;
        sz = sz + Zj;
        snx = snx + ma;
        sny = sny + mb;
        snz = snz + mc;
        sg += B.gray ? B.gray[q] : 0u;
    }
    if (count < k.min_num) return false;
    const double fc = (double)count;
    const float l = sqrtf((snx * snx + sny * sny) + snz * snz);
    o.x = sx / fc;
    o.y = sy / fc;
    o.z = sz / fc;
    o.nx = l > 0.f ? snx / l : 0.f;
    o.ny = l > 0.f ? sny / l : 0.f;
    o.nz = l > 0.f ? snz / l : 0.f;
    o.gray = (sg + (uint32_t)(count / 2)) / (uint32_t)count;
    return true;
}

// The points of image i at their pixels, a bit per pixel that makes one and
// the number of points per workgroup.
__global__ __launch_bounds__(256) void k_fuse3d(const Fuse3dView *__restrict__ V, int i, Fuse3dConst k,
                                                FusedPoint *__restrict__ out,
                                                unsigned long long *__restrict__ bits,
                                                int *__restrict__ counts)
{
    __shared__ int s_n[4];
    const long long p = (long long)blockIdx.x * 256 + threadIdx.x;
    FusedPoint o;
    const bool kept = p < (long long)V[i].W * V[i].H && fuse_pixel(V, i, k, p, o);
    if (kept) out[p] = o;
    const unsigned long long m = __ballot(kept);
    if ((threadIdx.x & 63) == 0) {
        bits[p >> 6] = m;
        s_n[threadIdx.x >> 6] = __popcll(m);
    }
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = (s_n[0] + s_n[1]) + (s_n[2] + s_n[3]);
}

// Exclusive sums of the n counts in place, and their total: one workgroup,
// 4096 counts a turn (one turn covers a megapixel).
__global__ __launch_bounds__(1024) void k_scan_counts(int *__restrict__ counts, int n, int *__restrict__ total)
{
    __shared__ int s_wave[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int carry = 0;
    for (int base = 0; base < n; base += 4096) {
        const int at = base + (int)threadIdx.x * 4;
        int v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = at + k < n ? counts[at + k] : 0;
        const int sum = (v[0] + v[1]) + (v[2] + v[3]);
        int run = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int below = __shfl_up(run, d);
            if (lane >= d) run += below;
        }
        if (lane == 63) s_wave[wave] = run;
        __syncthreads();
        int before = carry, all = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            if (w < wave) before += s_wave[w];
            all += s_wave[w];
        }
        before += run - sum;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (at + k < n) counts[at + k] = before;
            before += v[k];
        }
        carry += all;
        __syncthreads();                       // s_wave is written again
    }
    if (threadIdx.x == 0) *total = carry;
}

// The points in pixel order, split into the output arrays; those past room
// are counted only.  Bound by its launch and bytes: a view of about a megapixel
// with 116 thousand points takes 6.8 us, and the sums 4.9, where the library's
// select over (point, flag) pairs and a pass that split its output took 138
// and 5.  The call for eight such views: 3.25 -> 2.28 ms.
__global__ __launch_bounds__(256) void k_compact_fused(const FusedPoint *__restrict__ dense,
                                                       const unsigned long long *__restrict__ bits,
                                                       const int *__restrict__ offsets, long long room,
                                                       double *__restrict__ xyz, float *__restrict__ normal,
                                                       uint8_t *__restrict__ gray)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long *w = bits + (size_t)blockIdx.x * 4;
    const unsigned long long m = w[wave];
    if (!((m >> lane) & 1ull)) return;
    long long t = offsets[blockIdx.x] + __popcll(m & ((1ull << lane) - 1ull));
    for (int k = 0; k < wave; ++k) t += __popcll(w[k]);
    if (t >= room) return;
    const FusedPoint o = dense[(long long)blockIdx.x * 256 + threadIdx.x];
    xyz[3 * t] = o.x;
    xyz[3 * t + 1] = o.y;
    xyz[3 * t + 2] = o.z;
    normal[3 * t] = o.nx;
    normal[3 * t + 1] = o.ny;
    normal[3 * t + 2] = o.nz;
    gray[t] = (uint8_t)min(o.gray, 255u);
}

__device__ __forceinline__ float lower(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ float upper(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double lower(double a, double b) { return fmin(a, b); }
__device__ __forceinline__ double upper(double a, double b) { return fmax(a, b); }

// Batcher's odd-even merge sort of N registers (static indices only, any N;
// values are finite or infinite, no NaN: min and max order them).
template <typename T, int N>
__device__ __forceinline__ void sort_net(T (&v)[N])
{
#pragma unroll
    for (int p = 1; p < N; p <<= 1)
#pragma unroll
        for (int k = p; k >= 1; k >>= 1)
#pragma unroll
            for (int i = 0; i + k < N; ++i) {
                const int j = k % p;
                if (i >= j && (i - j) % (2 * k) < k && i / (2 * p) == (i + k) / (2 * p)) {
                    const T lo = lower(v[i], v[i + k]), hi = upper(v[i], v[i + k]);
                    v[i] = lo;
                    v[i + k] = hi;
                }
            }
}

template <typename T, int N>
__device__ __forceinline__ T median_sorted(const T (&v)[N], int n)
{
    T lo = v[0], hi = v[0];
#pragma unroll
    for (int i = 0; i <= N / 2; ++i) {
        if (i == (n - 1) / 2) lo = v[i];
        if (i == n / 2) hi = v[i];
    }
    return (n & 1) ? hi : (T)0.5 * (lo + hi);
}

// Decode + hole fill.  Output float (per-view DSM, then medianBlur) or double
// (proj_to_grid stand-alone).
template <typename OUT>
__global__ void k_decode_fill(const unsigned long long *__restrict__ cell_max, int e_size,
                              int n_size, OUT *__restrict__ dsm)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long long)e_size * n_size) return;
    const int r = (int)(i / e_size), c = (int)(i - (long long)r * e_size);
    const unsigned long long k = cell_max[i];
    if (k != 0ull) { dsm[i] = (OUT)dec_f64(k); return; }
    double v[9];
    int n = 0;
#pragma unroll
    for (int dr = -1; dr <= 1; ++dr)
#pragma unroll
        for (int dc = -1; dc <= 1; ++dc) {
            const int rr = r + dr, cc = c + dc;
            const int slot = (dr + 1) * 3 + (dc + 1);
            unsigned long long kk = 0ull;
            if (rr >= 0 && cc >= 0 && rr < n_size && cc < e_size) kk = cell_max[(size_t)rr * e_size + cc];
            v[slot] = kk ? dec_f64(kk) : (double)INFINITY;
            n += kk ? 1 : 0;
        }
    if (n == 0) { dsm[i] = (OUT)NAN; return; }
    sort_net<double, 9>(v);
    dsm[i] = (OUT)median_sorted<double, 9>(v, n);
}

// min, middle, max of three values (no NaN).
__device__ __forceinline__ void sort3(float &a, float &b, float &c)
{
    const float lo = __builtin_amdgcn_fmed3f(a, b, -INFINITY), hi = __builtin_amdgcn_fmed3f(a, b, INFINITY);
    a = __builtin_amdgcn_fmed3f(lo, c, -INFINITY);
    b = __builtin_amdgcn_fmed3f(lo, hi, c);
    c = __builtin_amdgcn_fmed3f(hi, c, INFINITY);
}

// 3x3 medians of R cells in a column from the R + 2 rows of three values
// around them, for the windows without NaN: each row is sorted once and serves
// the three windows it is in, whose median is the middle of (largest of the
// lowest, middle of the middle, lowest of the largest).  Bit r of the result:
// window r holds a NaN and takes median_of_window.
template <int R>
__device__ __forceinline__ uint32_t column_medians(const float (&w)[R + 2][3], float (&out)[R])
{
    float lo[R + 2], mi[R + 2], hi[R + 2];
    uint32_t nan = 0u;
#pragma unroll
    for (int r = 0; r < R + 2; ++r) {
        lo[r] = w[r][0]; mi[r] = w[r][1]; hi[r] = w[r][2];
        if (__builtin_isunordered(w[r][0], w[r][1]) || w[r][2] != w[r][2]) nan |= 7u << r;   // windows r - 2 .. r, shifted by 2
        sort3(lo[r], mi[r], hi[r]);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float a = __builtin_amdgcn_fmed3f(__builtin_amdgcn_fmed3f(lo[r], lo[r + 1], INFINITY), lo[r + 2], INFINITY);
        const float b = __builtin_amdgcn_fmed3f(mi[r], mi[r + 1], mi[r + 2]);
        const float c = __builtin_amdgcn_fmed3f(__builtin_amdgcn_fmed3f(hi[r], hi[r + 1], -INFINITY), hi[r + 2], -INFINITY);
        out[r] = __builtin_amdgcn_fmed3f(a, b, c);
    }
    return (nan >> 2) & ((1u << R) - 1u);
}

// Median of nine values: NaN excluded, even count -> mean of the two middle
// values, all NaN -> NaN.
__device__ __forceinline__ float median_of_window(const float (&x)[9])
{
    float v[9];
    int n = 0;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        v[k] = x[k] == x[k] ? x[k] : INFINITY;
        n += x[k] == x[k] ? 1 : 0;
    }
    if (n == 0) return NAN;
    sort_net<float, 9>(v);
    return median_sorted<float, 9>(v, n);
}

// 3x3 median, replicated border, NaN excluded, all-NaN -> NaN.  A thread
// takes kMedRows cells of a column (6554^2 cells: 345 -> 112 us).
constexpr int kMedRows = 4;

__global__ __launch_bounds__(256) void k_median3(const float *__restrict__ in, int e_size, int n_size,
                                                 unsigned int first, float *__restrict__ out)
{
    // one-dimensional grid from block `first` of the raster on: any number of rows
    const unsigned int across = ((unsigned int)e_size + 63u) / 64u, block = first + blockIdx.x;
    const int c = (int)(block % across) * 64 + (threadIdx.x & 63);
    const int r0 = ((int)(block / across) * 4 + (threadIdx.x >> 6)) * kMedRows;
    if (c >= e_size || r0 >= n_size) return;
    float w[kMedRows + 2][3], m[kMedRows];
#pragma unroll
    for (int r = 0; r < kMedRows + 2; ++r)
#pragma unroll
        for (int dc = -1; dc <= 1; ++dc) {
            const int rr = max((int)min((unsigned int)r0 + r, (unsigned int)n_size) - 1, 0);   // row r0 - 1 + r
            const int cc = min(max(c + dc, 0), e_size - 1);
            w[r][dc + 1] = in[(size_t)rr * e_size + cc];
        }
    const uint32_t nan = column_medians<kMedRows>(w, m);
#pragma unroll
    for (int r = 0; r < kMedRows; ++r) {
        if (!(nan >> r & 1u)) continue;
        const float x[9] = {w[r][0], w[r][1], w[r][2], w[r + 1][0], w[r + 1][1], w[r + 1][2],
                            w[r + 2][0], w[r + 2][1], w[r + 2][2]};
        m[r] = median_of_window(x);
    }
#pragma unroll
    for (int r = 0; r < kMedRows; ++r)
        if (r0 + r < n_size) out[(size_t)(r0 + r) * e_size + c] = m[r];
}

// Per-view DSM in one pass over a tile of kVT_W x kVT_H cells: decode the
// cell keys, fill each empty cell with the median of its non-empty 3x3
// neighbours (the unfilled keys, as k_decode_fill), then the 3x3 median of
// the filled values (replicated border, NaN excluded, as k_median3) into
// `out`.  The heights of the tile and a 2-cell halo and the filled values of
// the tile and a 1-cell halo sit in LDS, at the same indices, so each key is
// read and decoded once per tile instead of by three kernels.  The tile's
// cells of `clear` (the other key grid, which the next view rasterises into)
// are zeroed; `keys` and `clear` must differ, since other tiles read this
// tile's keys as their halo.
//
// VALU issue is 87 % busy, and the 39 bytes a cell moved (tile halos, partial
// lines) run at 76 % of a copy's rate, so the rare work is listed and done by
// full waves: a wave of the tile nearly always holds an empty cell, and often a
// window with a NaN.  Where no lane of a wave has more than five neighbours (a
// grid finer than the pixels) the three largest of them hold the median, else
// all nine are sorted.  The medians share their rows' sorts (column_medians).
// 6554^2 cells of 0.3 m from 4096^2 pixels of 0.6 m: 789 -> 420 us.
constexpr int kVT_W = 64, kVT_H = 16;

__device__ __forceinline__ double min_f64(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));   // fmin would quieten its operands first
    return r;
}
__device__ __forceinline__ double max_f64(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Median of the n heights among v (the others are -inf), n > 0.  few: no lane
// of the wave has more than five.
__device__ __forceinline__ double median_of_heights(double (&v)[9], int n, bool few)
{
    double lo, hi;                             // the two middle ones (the same for an odd count)
    if (few) {
        double a = max_f64(v[0], v[1]), b = min_f64(v[0], v[1]), c = min_f64(b, v[2]);
        const double t = max_f64(b, v[2]);     // a >= b >= c: the largest so far
        b = min_f64(a, t);
        a = max_f64(a, t);
#pragma unroll
        for (int k = 3; k < 9; ++k) {
            const double p = min_f64(a, v[k]), q = min_f64(b, p);
            a = max_f64(a, v[k]);
            b = max_f64(b, p);
            c = max_f64(c, q);
        }
        // the n/2-th and (n-1)/2-th of n ascending, counted from the top
        hi = n >= 5 ? c : n >= 3 ? b : a;
        lo = n >= 4 ? c : n >= 2 ? b : a;
    } else {
        sort_net<double, 9>(v);                // the n heights are the last n
        lo = hi = v[8];
#pragma unroll
        for (int k = 4; k < 8; ++k) {
            if (k == 9 - n + (n - 1) / 2) lo = v[k];
            if (k == 9 - n + n / 2) hi = v[k];
        }
    }
    return (n & 1) ? hi : 0.5 * (lo + hi);
}

__global__ void __launch_bounds__(256) k_view_dsm(const unsigned long long *__restrict__ keys,
                                                  unsigned long long *__restrict__ clear, int e_size,
                                                  int n_size, float *__restrict__ out)
{
    constexpr int KW = kVT_W + 4, KH = kVT_H + 4;
    constexpr double kEmpty = -(double)INFINITY;
    __shared__ double sk[KH * KW];             // heights, -inf where empty
    __shared__ float sf[KH * KW];              // filled values, NaN where there is none
    __shared__ unsigned short list[KH * KW];   // empty cells, then windows with a NaN
    __shared__ int n_holes, n_windows;
    const int c0 = blockIdx.x * kVT_W, r0 = blockIdx.y * kVT_H;
    if (threadIdx.x == 0) { n_holes = 0; n_windows = 0; }
    __syncthreads();
    auto load = [&](int ky, int kx) {
        const int t = ky * KW + kx;
        const int r = r0 - 2 + ky, c = c0 - 2 + kx;
        unsigned long long k = 0ull;
        const bool inside = r >= 0 && c >= 0 && r < n_size && c < e_size;
        if (inside) k = keys[(size_t)r * e_size + c];
        const double z = k ? dec_f64(k) : kEmpty;
        sk[t] = z;
        if (k) sf[t] = (float)z;
        else if (inside && ky > 0 && ky < KH - 1 && kx > 0 && kx < KW - 1)
            list[atomicAdd(&n_holes, 1)] = (unsigned short)t;
    };
    // a wave takes 64 columns of every fourth row; the last four columns follow
    for (int ky = threadIdx.x >> 6; ky < KH; ky += 4) load(ky, threadIdx.x & 63);
    if (threadIdx.x < 4 * KH) load(threadIdx.x >> 2, 64 + (threadIdx.x & 3));
    __syncthreads();
    for (int h = threadIdx.x; h < n_holes; h += 256) {
        const int at = list[h];
        double v[9];
        int n = 0;
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            v[k] = sk[at + (k / 3 - 1) * KW + k % 3 - 1];
            n += v[k] != kEmpty ? 1 : 0;
        }
        const double z = median_of_heights(v, n, __ballot(n > 5) == 0ull);
        sf[at] = n ? (float)z : NAN;
    }
    __syncthreads();
    if (r0 == 0 || c0 == 0 || r0 + kVT_H >= n_size || c0 + kVT_W >= e_size) {
        // the median reads replicated borders: the ring of cells just outside
        for (int t = threadIdx.x; t < KH * KW; t += 256) {
            const int ky = t / KW, kx = t - ky * KW;
            const int r = r0 - 2 + ky, c = c0 - 2 + kx;
            if (r < -1 || c < -1 || r > n_size || c > e_size || (r >= 0 && c >= 0 && r < n_size && c < e_size)) continue;
            sf[t] = sf[(min(max(r, 0), n_size - 1) - r0 + 2) * KW + min(max(c, 0), e_size - 1) - c0 + 2];
        }
        __syncthreads();
    }
    constexpr int RT = kVT_H / 4;              // rows per thread
    const int tx = threadIdx.x & 63, ty = (threadIdx.x >> 6) * RT;
    const int c = c0 + tx;
    if (c < e_size) {
        float w[RT + 2][3], m[RT];
#pragma unroll
        for (int r = 0; r < RT + 2; ++r)
#pragma unroll
            for (int k = 0; k < 3; ++k) w[r][k] = sf[(ty + 1 + r) * KW + tx + 1 + k];
        const uint32_t nan = column_medians<RT>(w, m);
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            if (r0 + ty + r >= n_size) continue;
            const size_t i = (size_t)(r0 + ty + r) * e_size + c;
            clear[i] = 0ull;
            if (nan >> r & 1u) list[atomicAdd(&n_windows, 1)] = (unsigned short)((ty + r) * kVT_W + tx);
            else out[i] = m[r];
        }
    }
    __syncthreads();
    for (int h = threadIdx.x; h < n_windows; h += 256) {
        const int t = list[h], ky = t / kVT_W, kx = t % kVT_W;
        float x[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) x[k] = sf[(ky + 1 + k / 3) * KW + kx + 1 + k % 3];
        out[(size_t)(r0 + ky) * e_size + c0 + kx] = median_of_window(x);
    }
}

// Sorts a sequence that falls and then rises (with +inf at its end): one
// bitonic merge, the registers beyond N being +inf.
template <int N>
__device__ __forceinline__ void merge_valley(float (&v)[N])
{
    constexpr int M = N <= 8 ? 8 : N <= 16 ? 16 : N <= 32 ? 32 : 64;
#pragma unroll
    for (int j = M / 2; j > 0; j >>= 1)
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int l = i ^ j;
            if (l > i && l < N) {
                const float lo = fminf(v[i], v[l]), hi = fmaxf(v[i], v[l]);
                v[i] = lo;
                v[l] = hi;
            }
        }
}

// Cross-view fusion of a cell: median, median absolute deviation, mean of what
// lies within it.  N is the view count rounded up to 8, so a 40-view stack
// sorts 40 registers (305 comparators), not 64.  The deviations of the sorted
// values fall and then rise, so their median takes a merge, not a second sort
// (40 views of 6554^2 cells: 13.0 -> 3.3 ms with two 64-register bitonic sorts
// before, 2.1 TB/s of the stack).
template <int N>
__global__ __launch_bounds__(256) void k_fuse_stack(const float *__restrict__ stack, int nviews, long long ncell,
                             int min_measurements, float *__restrict__ out)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncell) return;
    float v[N];
    int n = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        float x = k < nviews ? stack[(size_t)k * ncell + i] : NAN;
        const bool ok = x == x;
        n += ok ? 1 : 0;
        v[k] = ok ? x : INFINITY;
    }
    if (n < min_measurements || n == 0) { out[i] = NAN; return; }
    float s[N];
#pragma unroll
    for (int k = 0; k < N; ++k) s[k] = v[k];
    sort_net<float, N>(s);
    const float med = median_sorted<float, N>(s, n);
#pragma unroll
    for (int k = 0; k < N; ++k) s[k] = s[k] == INFINITY ? INFINITY : fabsf(s[k] - med);
    merge_valley<N>(s);
    const float mad = median_sorted<float, N>(s, n);
    double acc = 0.0;
    int m = 0;
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if (v[k] != INFINITY && !(fabsf(v[k] - med) > mad)) { acc += (double)v[k]; ++m; }
    }
    out[i] = m > 0 ? (float)(acc / (double)m) : NAN;
}

__global__ void k_fill_u32(unsigned int *p, long long n, unsigned int v)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}
__global__ void k_fill_u64n(unsigned long long *p, long long n, unsigned long long v)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

static inline unsigned int nblk(long long n, int b) { return (unsigned int)((n + b - 1) / b); }

hipError_t launch_rasterize_view(const float *depth, int W, int H, const double *invP4_dev,
                                 DsmGridDev g, const vsm_geo_frame *geo,
                                 unsigned long long *cell_max, hipStream_t st)
{
    const dim3 grid((unsigned)((W + 63) / 64), (unsigned)((H + 3) / 4));
    if (geo) k_rasterize_view<true><<<grid, 256, 0, st>>>(depth, W, H, invP4_dev, g, *geo, cell_max);
    else k_rasterize_view<false><<<grid, 256, 0, st>>>(depth, W, H, invP4_dev, g, vsm_geo_frame{}, cell_max);
    return hipGetLastError();
}

hipError_t launch_fuse3d(const Fuse3dView *views, int i, int W, int H, Fuse3dConst k, long long room,
                         const Fuse3dScratch &f, hipStream_t st)
{
    const long long n = (long long)W * H;
    if (n <= 0) return hipSuccess;
    const unsigned nb = nblk(n, 256);
    k_fuse3d<<<nb, 256, 0, st>>>(views, i, k, f.dense, f.bits, f.counts);
    k_scan_counts<<<1, 1024, 0, st>>>(f.counts, (int)nb, f.total);
    if (room > 0) k_compact_fused<<<nb, 256, 0, st>>>(f.dense, f.bits, f.counts, room, f.xyz, f.normal, f.gray);
    return hipGetLastError();
}

hipError_t launch_enu_to_utm(const double *enu, long long n, const vsm_geo_frame &geo, double *out,
                             hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    k_enu_to_utm<<<nblk(n, 256), 256, 0, st>>>(enu, n, geo, out);
    return hipGetLastError();
}

hipError_t launch_rasterize_points(const double *pts, long long n, DsmGridDev g,
                                   unsigned long long *cell_max, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    k_rasterize_points<<<nblk(n, 256), 256, 0, st>>>(pts, n, g, cell_max);
    return hipGetLastError();
}

hipError_t launch_decode_fill_f32(const unsigned long long *cell_max, int e_size, int n_size,
                                  float *dsm, hipStream_t st)
{
    k_decode_fill<float><<<nblk((long long)e_size * n_size, 256), 256, 0, st>>>(cell_max, e_size,
                                                                             n_size, dsm);
    return hipGetLastError();
}

hipError_t launch_decode_fill_f64(const unsigned long long *cell_max, int e_size, int n_size,
                                  double *dsm, hipStream_t st)
{
    k_decode_fill<double><<<nblk((long long)e_size * n_size, 256), 256, 0, st>>>(cell_max, e_size,
                                                                              n_size, dsm);
    return hipGetLastError();
}

hipError_t launch_view_dsm(const unsigned long long *keys, unsigned long long *clear, int e_size, int n_size,
                           float *out, hipStream_t st)
{
    if (keys == clear) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((e_size + kVT_W - 1) / kVT_W), (unsigned)((n_size + kVT_H - 1) / kVT_H));
    k_view_dsm<<<grid, 256, 0, st>>>(keys, clear, e_size, n_size, out);
    return hipGetLastError();
}

hipError_t launch_median3(const float *in, int e_size, int n_size, float *out, hipStream_t st)
{
    // A launch holds fewer than 2^32 threads.  Blocks are 64 columns wide and 16
    // rows high, so a raster that is narrower or lower has more threads than
    // cells (2^28 rows of up to 8 cells and 2^30 columns of up to 2 reach the
    // limit) and takes several launches.
    constexpr unsigned int kMaxBlocks = 1u << 23;
    const unsigned int blocks = nblk(e_size, 64) * nblk(n_size, 4 * kMedRows);
    for (unsigned int first = 0; first < blocks; first += kMaxBlocks) {
        k_median3<<<std::min(kMaxBlocks, blocks - first), 256, 0, st>>>(in, e_size, n_size, first, out);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_fuse_stack(const float *stack, int nviews, long long ncell, int min_measurements,
                             float *out, hipStream_t st)
{
    if (nviews > 64) return hipErrorInvalidValue;
    void (*fn)(const float *, int, long long, int, float *) = nullptr;
    switch ((nviews + 7) / 8) {
    case 0:
    case 1: fn = k_fuse_stack<8>; break;
    case 2: fn = k_fuse_stack<16>; break;
    case 3: fn = k_fuse_stack<24>; break;
    case 4: fn = k_fuse_stack<32>; break;
    case 5: fn = k_fuse_stack<40>; break;
    case 6: fn = k_fuse_stack<48>; break;
    case 7: fn = k_fuse_stack<56>; break;
    default: fn = k_fuse_stack<64>; break;
    }
    fn<<<nblk(ncell, 256), 256, 0, st>>>(stack, nviews, ncell, min_measurements, out);
    return hipGetLastError();
}

hipError_t launch_fill_u32(unsigned int *p, long long n, unsigned int v, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    k_fill_u32<<<nblk(n, 256), 256, 0, st>>>(p, n, v);
    return hipGetLastError();
}

hipError_t launch_fill_u64n(unsigned long long *p, long long n, unsigned long long v,
                            hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    k_fill_u64n<<<nblk(n, 256), 256, 0, st>>>(p, n, v);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Allocation-free rasteriser.  Its only scratch, the per-cell 64-bit max keys,
// is this file-scope device array (each device holds its own copy for the
// life of the process).  Host code never passes the symbol itself to a kernel:
// it uses the device address taken once per device by scratch_init.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned long long scratch[kNoAllocMaxCells];

static std::mutex g_scratch_mu;
static std::vector<unsigned long long *> g_scratch_ptr;   // per device ordinal

hipError_t scratch_init(int device)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if ((int)g_scratch_ptr.size() <= device) g_scratch_ptr.resize(device + 1, nullptr);
    if (g_scratch_ptr[device]) return hipSuccess;
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device) return hipErrorInvalidDevice;      // the caller makes `device` current
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[device] = static_cast<unsigned long long *>(p);
    return hipSuccess;
}

hipError_t proj_to_grid_noalloc(int device, const double *pts, long long n, DsmGridDev g,
                                double *dsm, hipStream_t st)
{
    unsigned long long *cells = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (device >= 0 && device < (int)g_scratch_ptr.size()) cells = g_scratch_ptr[device];
    }
    if (!cells) return hipErrorNotInitialized;
    const long long ncell = (long long)g.e_size * g.n_size;
    if (ncell <= 0 || ncell > kNoAllocMaxCells) return hipErrorInvalidValue;
    // the previous call's keys are still there: clear this call's cells
    hipError_t e = launch_fill_u64n(cells, ncell, 0ull, st);
    if (e == hipSuccess) e = launch_rasterize_points(pts, n, g, cells, st);
    if (e == hipSuccess) e = launch_decode_fill_f64(cells, g.e_size, g.n_size, dsm, st);
    return e;
}

}  // namespace vsm
