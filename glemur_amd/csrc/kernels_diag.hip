// Mesh and error diagnostics of src/diagnostics.cu:33-110 and
// src/maths.cu:204-380,443-640: signed cell volume, octant wedge minimum,
// convexity, |B - ez| and |x - x_analytic| RMS errors, and the force-free
// parameter spread epsilon* along the central field line.  Positions are
// read in either precision (FP64, or FP32 hi + lo); per-point values are
// optionally stored for dumps, and the reductions are block partials summed
// or minimised in a fixed order.
#include "gm_device.hpp"

namespace gmd {
namespace {

constexpr int kB = 256;

// Positions in the precision of R: FP64 component arrays, or FP32 (hi, lo)
// triples.  Resolved at compile time: with a test per load the loads of the
// neighbours waited for one another.
template <class R>
struct PosRef {
    const R *x;
    const float *lo;
    long long P;
    __device__ void at(long long a, double v[3]) const
    {
        for (int c = 0; c < 3; ++c)
            if constexpr (sizeof(R) == 8) v[c] = x[c * P + a];
            else v[c] = (double)x[3 * a + c] + (double)lo[3 * a + c];
    }
};

__device__ inline double dot3(const double *a, const double *b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]; }
__device__ inline void cross3d(const double *a, const double *b, double *c)
{
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

// One inner point, x0 at padded offset a, zm and zp the positions below and
// above it: the 8 octant wedge products of the edges to
// the face neighbours (src/maths.cu:497-570), oriented so that an
// undistorted cell is positive; convexity -1 when any is negative
// (src/maths.cu:573-640); the forward-difference cell volume
// (src/maths.cu:443-494).
template <class R>
__device__ void mesh_point(const Geo &g, const PosRef<R> &X, long long a, const double x0[3], const double zm[3],
                           const double zp[3], double &wmin, double &conv, double &vol)
{
    double xm[3][2][3];
    X.at(a - 1, xm[0][0]);
    X.at(a + 1, xm[0][1]);
    X.at(a - g.sx, xm[1][0]);
    X.at(a + g.sx, xm[1][1]);
    for (int c = 0; c < 3; ++c) {
        xm[2][0][c] = zm[c];
        xm[2][1][c] = zp[c];
    }
    for (int d = 0; d < 3; ++d)
        for (int s = 0; s < 2; ++s)
            for (int c = 0; c < 3; ++c) xm[d][s][c] -= x0[c];
    wmin = 0;
    conv = 1;
    for (int u = 0; u < 2; ++u)
        for (int v = 0; v < 2; ++v)
            for (int w = 0; w < 2; ++w) {
                double cr[3];
                cross3d(xm[0][u], xm[1][v], cr);
                double wc = dot3(cr, xm[2][w]);
                const int s = 2 * (u + v + w);       // the reference's u+v+w
                if (s == 0 || s == 4) wc = -wc;
                if (s == 0 || wc < wmin) wmin = wc;
                if (wc < 0) conv = -1;
            }
    double cr[3];
    cross3d(xm[0][1], xm[1][1], cr);
    vol = dot3(cr, xm[2][1]);
}

// The joining operation of row quantity q (NaN-blind, as findDevMax) and
// the value it starts from
__device__ inline double row_join(int q, double a, double b)
{
    if (q == 0 || q == 8 || q == 9) return a + b;
    if (q == 6 || q == 7) return b < a ? b : a;
    return nb_max(a, b);
}
__device__ inline double row_start(int q) { return q == 6 ? 1.0 : q == 7 ? 1e300 : 0.0; }
__device__ inline double wave_min(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double u = __shfl_xor(v, o, 64);
        v = u < v ? u : v;
    }
    return v;
}

// Everything a time-series row reduces over the inner points, in one pass.
//  - diag: energy density |B|^2 det / 2^(#boundary faces)
//    (src/maths.cu:647-680), |J|, |JxB|/|B|^2 (src/maths.cu:168-200) and
//    |JxB|/(|J||B|) (0/0 := 0), and the maxima of |JxB| and |J||B| (their
//    quotient is the relaxation criterion);
//  - mesh: convexity and wedge minimum (mesh_point);
//  - errs: |B - ez|^2 (src/maths.cu:294-330) and |x - x_an|^2
//    (src/maths.cu:334-377);
//  - eps: epsilon* (src/maths.cu:204-290): along the column i = nx/2,
//    j = ny/2, a_k = J.B / B^2 and z_k = z of the position; the maximum over
//    all pairs of sqrt2 |a_n - a_k| / |z_n - z_k| (pairs with equal z count
//    0), by neps further workgroups of 16 rows k each.
// Bound by memory: 56 bytes a point in FP32 (positions 24, B 12, J 12, det
// 8), read once here and three times by a pass per quantity.  A thread
// marches KZ planes of one column, so its z neighbours stay in registers
// and the index divisions are done once; the other neighbours hit in cache.
// 129 x 129 x 385 (FP32, all quantities): 0.18 ms in one launch, 2.0 TB/s,
// against 0.6 ms in four launches of 512 workgroups, one wave of them
// summing their partials serially; what is left is FP64 arithmetic.
// Partials of a workgroup go to part[q * nb + block], q = energy, |J|max,
// the four other maxima, convexity, wedge, and the two error sums.
constexpr int kQ = 10, kRowBlocks = 2048, kEpsRows = 16;

template <class R>
struct RowArgs {
    Geo g;
    PosRef<R> X;
    const double *det;
    double ar, az, phi1;
    int diag, mesh, errs, eps;
    double *cellVol, *convex, *wedge;
    int nb, bx, G, KZ, neps;  // workgroups over points (bx per layer of G KZ planes), and of epsilon*
    double *part;
};

// The columns t, t + bx kB, ... < nx ny and planes [k0, k1) of a thread of
// workgroup blk.  Where a workgroup has more threads than the grid columns, G
// groups of them take the planes in turn (2 x 2 x 50000, a row with the mesh and
// error quantities in FP32: 191 us without, 35 with).
struct RowPart {
    int t, k0, k1;
};
template <class R>
__device__ RowPart row_part(const RowArgs<R> &A, int blk)
{
    const int layer = blk / A.bx, nxy = A.g.nx * A.g.ny;
    RowPart p;
    int sub = 0;
    p.t = (blk - layer * A.bx) * kB + threadIdx.x;
    if (A.G > 1) {
        sub = threadIdx.x / nxy;
        p.t = sub < A.G ? threadIdx.x - sub * nxy : nxy;
    }
    p.k0 = (layer * A.G + sub) * A.KZ;
    p.k1 = min(p.k0 + A.KZ, A.g.nz);
    if (p.k0 >= p.k1) p.t = nxy;
    return p;
}

template <class R>
__device__ void eps_star_rows(const RowArgs<R> &A, const R *B, const R *J, int blk)
{
    const Geo &g = A.g;
    __shared__ double zr[kEpsRows], ar[kEpsRows], red[kB / 64];
    auto column = [&](int k, double &z, double &al) {
        const long long a = gidx(g, g.nx / 2 + 1, g.ny / 2 + 1, k + 1);
        const double b[3] = {(double)B[a], (double)B[g.P + a], (double)B[2 * g.P + a]};
        const double jj[3] = {(double)J[a], (double)J[g.P + a], (double)J[2 * g.P + a]};
        al = dot3(jj, b) / dot3(b, b);
        double p[3];
        A.X.at(a, p);
        z = p[2];
    };
    const int k0 = blk * kEpsRows, rows = min(kEpsRows, g.nz - k0);
    if ((int)threadIdx.x < rows) column(k0 + threadIdx.x, zr[threadIdx.x], ar[threadIdx.x]);
    __syncthreads();
    const double SQRT2 = 1.414213562373095;   // the reference's literal (src/global.h:18)
    double m = 0;
    for (int n = threadIdx.x; n < g.nz; n += kB) {
        double zn, an;
        column(n, zn, an);
        for (int r = 0; r < rows; ++r)
            if (zn != zr[r]) {
                const double v = SQRT2 * fabs((an - ar[r]) / (zn - zr[r]));
                if (v > m) m = v;
            }
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < kB / 64; ++q) m = nb_max(m, red[q]);
        A.part[kQ * A.nb + blk] = m;
    }
}

// errB and errXb of the columns of workgroup blk
template <class R>
__device__ void errs_block(const RowArgs<R> &A, const R *B, int blk)
{
    const Geo &g = A.g;
    const RowPart part = row_part(A, blk);
    const int k0 = part.k0, k1 = part.k1, nxy = g.nx * g.ny;
    double e1 = 0, e2 = 0;
    for (int t = part.t; t < nxy; t += A.bx * kB) {
        const int j = t / g.nx, i = t - j * g.nx;
        long long a = gidx(g, i + 1, j + 1, k0 + 1);
        const double x = i * g.dx + g.Ox, y = j * g.dy + g.Oy;
#pragma unroll 1
        for (int k = k0; k < k1; ++k, a += g.sxy) {
            double p[3], sf, cf;
            A.X.at(a, p);
            const double b0 = B[a], b1 = B[g.P + a], b2 = (double)B[2 * g.P + a] - 1.;
            e1 += b0 * b0 + b1 * b1 + b2 * b2;
            const double z = k * g.dz + g.Oz;
            const double f = exp(-(x * x + y * y) / (A.ar * A.ar) - z * z / (A.az * A.az)) * A.phi1;
            sincos(f, &sf, &cf);
            const double d0 = p[0] - cf * x - sf * y;
            const double d1 = p[1] + sf * x - cf * y;
            const double d2 = p[2] - z;
            e2 += d0 * d0 + d1 * d1 + d2 * d2;
        }
    }
    __shared__ double red[2][kB / 64];
    const double s1 = wave_sum(e1), s2 = wave_sum(e2);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = s1;
        red[1][threadIdx.x >> 6] = s2;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double v = 0;
        for (int s = 0; s < kB / 64; ++s) v += red[threadIdx.x][s];
        A.part[(8 + threadIdx.x) * A.nb + blk] = v;
    }
}

// EXTRA: more than the diag quantities is wanted.  With errs every workgroup
// of points has a second one for the two error sums, eight further on (the
// same XCD, whose L2 then holds the positions and B): the exponential and
// angle functions bind the vector units while the rest waits for memory, but
// in one thread their constants cost it half the waves.
template <class R, bool EXTRA>
__global__ void __launch_bounds__(kB, sizeof(R) == 8 ? 3 : 4) k_row(RowArgs<R> A, const R *B, const R *J)
{
    // the few workgroups of epsilon* first, their chain is the longest
    if ((int)blockIdx.x < A.neps) return eps_star_rows(A, B, J, blockIdx.x);
    int blk = blockIdx.x - A.neps;
    if (EXTRA && A.errs) {
        const bool main = A.diag || A.mesh, second = blk >> 3 & 1;
        if (main) blk = (blk >> 4) * 8 + (blk & 7);
        if (blk >= A.nb) return;
        if (!main || second) return errs_block(A, B, blk);
    }
    const Geo &g = A.g;
    const RowPart part = row_part(A, blk);
    const int k0 = part.k0, k1 = part.k1, nxy = g.nx * g.ny;
    double e = 0, jm = 0, r1 = 0, r2 = 0, r3 = 0, r4 = 0, cm = 1, wm = 1e300;
    for (int t = part.t; t < nxy; t += A.bx * kB) {
        const int j = t / g.nx, i = t - j * g.nx;
        const int bxy = (i == 0) + (j == 0) + (i == g.nx - 1) + (j == g.ny - 1);
        long long a = gidx(g, i + 1, j + 1, k0 + 1);
        const long long t0 = (long long)nxy * k0 + t;
        double xm[3], x0[3], xp[3];
        if (EXTRA && A.mesh) {
            A.X.at(a, x0);
            A.X.at(a - g.sxy, xm);
        }
#pragma unroll 1
        for (int k = k0; k < k1; ++k, a += g.sxy) {
            if (A.diag) {
                const double b[3] = {(double)B[a], (double)B[g.P + a], (double)B[2 * g.P + a]};
                const double jj[3] = {(double)J[a], (double)J[g.P + a], (double)J[2 * g.P + a]};
                const double b2 = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
                e += ldexp(b2 * A.det[a], -(bxy + (k == 0) + (k == g.nz - 1)));
                double c[3];
                cross3(jj, b, c);
                const double nc = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
                const double nj = sqrt(jj[0] * jj[0] + jj[1] * jj[1] + jj[2] * jj[2]);
                const double den = nj * sqrt(b2);
                jm = nb_max(jm, nj);
                r1 = nb_max(r1, nc / b2);
                r2 = nb_max(r2, den > 0 ? nc / den : 0.0);
                r3 = nb_max(r3, nc);
                r4 = nb_max(r4, den);
            }
            if (!EXTRA || !A.mesh) continue;
            double w, c, v;
            A.X.at(a + g.sxy, xp);
            mesh_point(g, A.X, a, x0, xm, xp, w, c, v);
            const long long at = t0 + (long long)nxy * (k - k0);
            if (A.cellVol) A.cellVol[at] = v;
            if (A.convex) A.convex[at] = c;
            if (A.wedge) A.wedge[at] = w;
            wm = w < wm ? w : wm;
            cm = c < cm ? c : cm;
            for (int q = 0; q < 3; ++q) { xm[q] = x0[q]; x0[q] = xp[q]; }
        }
    }
    __shared__ double red[kQ][kB / 64];
    const int w = threadIdx.x >> 6;
    auto put = [&](int q, double v) { if ((threadIdx.x & 63) == 0) red[q][w] = v; };
    if (A.diag) {
        put(0, wave_sum(e));
        put(1, wave_max(jm));
        put(2, wave_max(r1));
        put(3, wave_max(r2));
        put(4, wave_max(r3));
        put(5, wave_max(r4));
    }
    if (EXTRA) {
        put(6, wave_min(cm));
        put(7, wave_min(wm));
    }
    __syncthreads();
    if ((int)threadIdx.x < (EXTRA ? 8 : 6)) {
        const int q = threadIdx.x;
        double v = red[q][0];
        for (int s = 1; s < kB / 64; ++s) v = row_join(q, v, red[q][s]);
        A.part[q * A.nb + blk] = v;
    }
}

// out[0..5] the diag quantities, out[8] min convexity, out[9] min wedge,
// out[10] errB_1ez, out[11] errXb_XbAn, out[12] epsilon*: a wave each
template <class R>
__global__ void __launch_bounds__(64 * (kQ + 1)) k_row_final(RowArgs<R> A, long long N, double *out)
{
    const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (q < 6 ? !A.diag : q < 8 ? !A.mesh : q < kQ ? !A.errs : !A.eps) return;
    const int n = q < kQ ? A.nb : A.neps;
    const double *p = A.part + q * A.nb;
    double v = row_start(q);
    for (int i = lane; i < n; i += 64 * 8) {   // eight loads in flight a lane
        double u[8];
        for (int r = 0; r < 8; ++r) u[r] = p[min(i + 64 * r, n - 1)];
        for (int r = 0; r < 8; ++r) v = row_join(q, v, i + 64 * r < n ? u[r] : row_start(q));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = row_join(q, v, __shfl_xor(v, o, 64));
    if (lane != 0) return;
    if (q == 0) v = v * A.g.dx * A.g.dy * A.g.dz;
    if (q == 8 || q == 9) v = sqrt(v) / sqrt((double)N);
    out[q < 6 ? q : q + 2] = v;
}

}  // namespace

int row_parts() { return kQ * kRowBlocks + 3840 / kEpsRows; }

template <class R>
int launch_row(hipStream_t s, const Geo &g, const double *x64, const float *xh, const float *xl, const R *B, const R *J,
               const double *det, double ar, double az, double phi1, int diag, int mesh, int errs, int eps,
               double *cellVol, double *convex, double *wedge, double *part, double *out)
{
    if (eps && g.nz > 3840) return -1;
    const bool maps = cellVol || convex || wedge, extra = mesh || errs || maps;
    PosRef<R> X{nullptr, xl, g.P};
    if constexpr (sizeof(R) == 8) X.x = x64;
    else X.x = xh;
    RowArgs<R> A{g, X, det, ar, az, phi1, diag, mesh || maps, errs, eps, cellVol, convex, wedge,
              0, 0, 0, 0, 0, part};
    // as many planes a thread as leave at most kRowBlocks workgroups: one on
    // small grids (more workgroups), 13 at 129 x 129 x 385.  Twice as many
    // workgroups keep the kernel that joins their partials busy longer than
    // they save (a row of 100^3 points in FP32 40 us against 30, 129 x 129 x
    // 385 67 against 62)
    const long long nxy = (long long)g.nx * g.ny, cols = (nxy + kB - 1) / kB;
    A.bx = (int)(cols < kRowBlocks ? cols : kRowBlocks);
    A.G = nxy < kB ? (int)(kB / nxy) : 1;
    const int layers = kRowBlocks / A.bx * A.G;
    A.KZ = (g.nz + layers - 1) / layers;
    A.nb = diag || extra ? A.bx * ((g.nz + A.G * A.KZ - 1) / (A.G * A.KZ)) : 0;
    A.neps = eps ? (g.nz + kEpsRows - 1) / kEpsRows : 0;
    const bool two = errs && (diag || A.mesh);
    const dim3 grid(A.neps + (two ? 2 * ((A.nb + 7) / 8 * 8) : A.nb));
    if (extra)
        hipLaunchKernelGGL((k_row<R, true>), grid, dim3(kB), 0, s, A, B, J);
    else
        hipLaunchKernelGGL((k_row<R, false>), grid, dim3(kB), 0, s, A, B, J);
    A.mesh = mesh;
    if (out)
        hipLaunchKernelGGL(k_row_final<R>, dim3(1), dim3(64 * (kQ + 1)), 0, s, A, (long long)g.nx * g.ny * g.nz, out);
    return 0;
}
template int launch_row<double>(hipStream_t, const Geo &, const double *, const float *, const float *, const double *,
                                const double *, const double *, double, double, double, int, int, int, int, double *,
                                double *, double *, double *, double *);
template int launch_row<float>(hipStream_t, const Geo &, const double *, const float *, const float *, const float *,
                               const float *, const double *, double, double, double, int, int, int, int, double *,
                               double *, double *, double *, double *);

}  // namespace gmd
