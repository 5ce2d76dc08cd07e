// Device helpers shared by the fused stage kernels (FP64 and FP32).
#pragma once

#include "gm_device.hpp"
#include "gm_fused.hpp"

namespace gmd {
namespace {

// Workgroup id -> logical tile so that the blocks one XCD receives
// (hardware deals ids round-robin over the 8 XCDs) form a contiguous range
// of tiles and share halos in that XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int nb)
{
    int q = nb >> 3, r = nb & 7;
    int x = bid & 7, w = bid >> 3;
    int base = x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q;
    return base + w;
}

// The inverse of xcd_remap: the workgroup index that xcd_remap sends to
// logical index L among nb.
__device__ __forceinline__ int xcd_unremap(int L, int nb)
{
    const int q = nb >> 3, r = nb & 7, head = r * (q + 1);
    int x, w;
    if (L < head) {
        x = L / (q + 1);
        w = L - x * (q + 1);
    } else {   // q > 0 here: L < nb = 8q + r
        x = r + (L - head) / q;
        w = L - head - (x - r) * q;
    }
    return w * 8 + x;
}

// Two-sum (Knuth): s + e == a + b exactly.
__device__ __forceinline__ void two_sum(float a, float b, float &s, float &e)
{
    s = a + b;
    float bb = s - a;
    e = (a - (s - bb)) + (b - bb);
}

__device__ __forceinline__ int nface(const Geo &g, int face) { return face == 0 ? g.ny : g.nx; }

// B and det at a line-tied ghost-face point from its first inner neighbour
// x_in along the normal and the precomputed constants (src/boundaries.cu:
// 164-186): jac = [normal column from x_in and the outer ghost | tangential
// columns], B_normal = B0_normal.
// (FACE: the face as a compile-time constant, so that no array is indexed
// at run time)
template <int FACE>
__device__ __forceinline__ void ghost_b_f(const Geo &g, const GhostPt &G, int side, const double xin[3],
                                         double B[3], double &det)
{
    const double h1 = FACE == 0 ? g.dx1 : FACE == 1 ? g.dy1 : g.dz1;
    constexpr int t0 = FACE == 0 ? 1 : 0, t1 = FACE == 2 ? 1 : 2;
    double jac[3][3], d[3];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        d[l] = side ? G.x2[l] - xin[l] : xin[l] - G.x2[l];
        jac[l][t0] = G.tc0[l];
        jac[l][t1] = G.tc1[l];
    }
    jac_col(jac, FACE, d, h1);
    double detJac1 = cauchy_b(jac, G.b0, FACE, B);
    det = 1 / detJac1;
}
__device__ __forceinline__ void ghost_b(const Geo &g, const GhostPt &G, int face, int side, const double xin[3],
                                       double B[3], double &det)
{
    if (face == 0) ghost_b_f<0>(g, G, side, xin, B, det);
    else if (face == 1) ghost_b_f<1>(g, G, side, xin, B, det);
    else ghost_b_f<2>(g, G, side, xin, B, det);
}

// floor(v / n) of 0 <= v < 2^20, n > 0 with inv = 1 / n to an ulp: (v + 1/2) / n
// is at least 1/(2n) away from a whole number, and inv's error and the
// product's rounding move it by at most (v + 1/2) 2^-22 / n, which is less
// while v + 1/2 < 2^21
__device__ __forceinline__ int small_div(int v, float inv) { return (int)(((float)v + 0.5f) * inv); }

// The points of a block launch a thread computes: output point and face
// neighbour of a bw x bh x bd block, in box coordinates (the block starts at
// 2); threads without one repeat the last.
struct BlockRole {
    bool own, ring;
    int oc, orr, oz, rc, rr, rz;
};
__device__ __forceinline__ BlockRole block_role(int t, int bw, int bh, int bd)
{
    BlockRole b;
    const float iw = __builtin_amdgcn_rcpf((float)bw), ih = __builtin_amdgcn_rcpf((float)bh);
    const int np = bw * bh * bd, fx = bh * bd, fy = bw * bd, fz = bw * bh, nr = 2 * (fx + fy + fz);
    b.own = t < np;
    b.ring = t < nr;
    const int v = min(t, np - 1), vy = small_div(v, iw), vz = small_div(vy, ih);
    b.oc = 2 + v - vy * bw;
    b.orr = 2 + vy - vz * bh;
    b.oz = 2 + vz;
    // faces x- x+ y- y+ z- z+
    int u = min(t, nr - 1);
    const int axis = u < 2 * fx ? 0 : u < 2 * (fx + fy) ? 1 : 2;
    u -= axis == 0 ? 0 : axis == 1 ? 2 * fx : 2 * (fx + fy);
    const int f = axis == 0 ? fx : axis == 1 ? fy : fz, s = u >= f;
    u -= s * f;
    const int q = small_div(u, axis == 0 ? ih : iw), p = u - q * (axis == 0 ? bh : bw);   // first and second tangent
    b.rc = axis == 0 ? (s ? bw + 2 : 1) : 2 + p;
    b.rr = axis == 1 ? (s ? bh + 2 : 1) : 2 + (axis == 0 ? p : q);
    b.rz = axis == 2 ? (s ? bd + 2 : 1) : 2 + q;
    return b;
}

// Wave reductions by lane shifts within the vector registers (rows of 16,
// then across rows); the result is in lane 63.  Values >= 0 for the maxima.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp0(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false); }
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp0(float v) { return __builtin_bit_cast(float, dpp0<CTRL, ROWS>(__builtin_bit_cast(int, v))); }
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp0(double v)
{
    const long long b = __builtin_bit_cast(long long, v);
    const unsigned lo = dpp0<CTRL, ROWS>((int)b), hi = dpp0<CTRL, ROWS>((int)(b >> 32));
    return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}
template <class R, class F>
__device__ __forceinline__ R wave_reduce63(R v, F f)
{
    v = f(v, dpp0<0x111, 0xf>(v));   // row_shr 1, 2, 4, 8
    v = f(v, dpp0<0x112, 0xf>(v));
    v = f(v, dpp0<0x114, 0xf>(v));
    v = f(v, dpp0<0x118, 0xf>(v));
    v = f(v, dpp0<0x142, 0xa>(v));   // row_bcast 15 into rows 1 and 3
    v = f(v, dpp0<0x143, 0xc>(v));   // row_bcast 31 into rows 2 and 3
    return v;
}
template <class R>
__device__ __forceinline__ R wave_max63(R v) { return wave_reduce63(v, [](R a, R b) { return b > a ? b : a; }); }
template <class R>
__device__ __forceinline__ R wave_sum63(R v) { return wave_reduce63(v, [](R a, R b) { return a + b; }); }

}  // namespace
}  // namespace gmd
