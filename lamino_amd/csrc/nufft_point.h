// Placement of the polar grids' points on the fine grid and the exchange between a
// half-set point and its mirror, shared by every kernel that visits points.
#pragma once
#include "common.h"
#include "nufft.h"

namespace lam {

inline constexpr double kTwoPi = 6.283185307179586476925286766559;

__device__ __forceinline__ int wrapi(int i, int n) {
    if (i < 0) i += n;
    else if (i >= n) i -= n;
    return i;
}

// Coordinate arithmetic is kept free of FMA contraction so that every kernel
// that places a point (binning, spreading, interpolation) computes bitwise the
// same fine coordinate and first kernel cell.

// Folds t into one period and returns the first kernel cell ceil(t - W/2).
// The fold multiplies by the reciprocal 1/nf: at an exact multiple of nf it
// may land on -0 ulp or nf, which every caller wraps (wrap0) identically.
__device__ __forceinline__ int first_cell(double &t, double nf, double rnf, int W) {
#pragma clang fp contract(off)
    const double fl = floor(t * rnf);
    t -= fl * nf;
    return (int)ceil(t - 0.5 * W);
}

// ES kernel weights for one axis: cells i0 .. i0+W-1 around the folded coordinate t.
template <int W>
__device__ __forceinline__ void es_weights(double t, int i0, float beta, float *wts) {
    const float z0 = (float)(((double)i0 - t) * (2.0 / W));
    const float dz = 2.0f / (float)W;
#pragma unroll
    for (int m = 0; m < W; ++m) {
        const float z = z0 + dz * (float)m;
        const float r = 1.0f - z * z;
        // r in (0, 1]: the hardware square root (no denormal rescaling needed)
        wts[m] = r > 0.f ? __expf(beta * (__builtin_amdgcn_sqrtf(r) - 1.0f)) : 0.f;
    }
}

// The same weights with the exponent's base 2 folded into beta (b2 = beta log2 e, one fused
// multiply-add per cell) and the edge test only where a cell can sit on the support's edge.
template <int W>
__device__ __forceinline__ void es_weights2(double t, int i0, float b2, float *wts) {
    const float z0 = (float)(((double)i0 - t) * (2.0 / W));
    const float dz = 2.0f / (float)W;
#pragma unroll
    for (int m = 0; m < W; ++m) {
        const float z = z0 + dz * (float)m;
        const float r = 1.0f - z * z;
        const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(b2, __builtin_amdgcn_sqrtf(r), -b2));
        wts[m] = (m > 0 && m < W - 1) || r > 0.f ? w : 0.f;
    }
}

struct PointFrame {
    double dX, dY, k0, j0, sx, sy, sz;  // qX step, qY step, centres, fine scales nf/(2 pi)
    double rx, ry, rz;                  // 1 / nf per axis
};

inline PointFrame point_frame(const Grid &g, const NufftPlan &pl) {
    PointFrame f;
    f.dX = kTwoPi / (double)g.C;
    f.dY = kTwoPi / (double)g.R;
    f.k0 = 0.5 * (double)(g.C - 1);
    f.j0 = 0.5 * (double)(g.R - 1);
    f.sx = (double)pl.nf[2] / kTwoPi;
    f.sy = (double)pl.nf[1] / kTwoPi;
    f.sz = (double)pl.nf[0] / kTwoPi;
    f.rx = 1.0 / (double)pl.nf[2];
    f.ry = 1.0 / (double)pl.nf[1];
    f.rz = 1.0 / (double)pl.nf[0];
    return f;
}

__device__ __forceinline__ void point_coords(const Geo &g, const PointFrame &f, int j, int k, double &tx, double &ty,
                                             double &tz) {
#pragma clang fp contract(off)
    const double qX = ((double)k - f.k0) * f.dX;
    const double qY = ((double)j - f.j0) * f.dY;
    tx = (qX * g.ux + qY * g.vx) * f.sx;
    ty = (qY * g.vy) * f.sy;
    tz = (qX * g.uz + qY * g.vz) * f.sz;
}

// Placement of one point: folded coordinates, first cells, weights.
template <int W>
struct Placed {
    int ix, iy, iz;
    float wx[W], wy[W], wz[W];
};

template <int W>
__device__ __forceinline__ void place(const Geo &g, const PointFrame &fr, int j, int k, int nfz, int nfy, int nfx,
                                      float beta, Placed<W> &pt) {
    double tx, ty, tz;
    point_coords(g, fr, j, k, tx, ty, tz);
    pt.ix = first_cell(tx, nfx, fr.rx, W);
    pt.iy = first_cell(ty, nfy, fr.ry, W);
    pt.iz = first_cell(tz, nfz, fr.rz, W);
    es_weights<W>(tx, pt.ix, beta, pt.wx);
    es_weights<W>(ty, pt.iy, beta, pt.wy);
    es_weights<W>(tz, pt.iz, beta, pt.wz);
}

__device__ __forceinline__ int wrap0(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// The value a half-set point spreads (times d_p): v = c(q) + conj c(-q) of plane p, from
// a = c(q) and b = c(-q) of the point's plane (the mirror is q's negative).  Paired planes
// hold Z = P2m + i P2m+1 in plane 2m: the even plane's value is Z(q) + conj Z(-q), the odd
// one's -i (Z(q) - conj Z(-q)); the centre point (its own mirror) takes Re Z or Im Z.
__device__ __forceinline__ float2 half_point_value(float2 a, float2 b, long long p, long long idx, long long S,
                                                   int paired) {
    const long long mir = S - 1 - idx;
    if (!paired) return mir != idx ? cadd(a, cconj(b)) : a;
    if (!(p & 1)) return mir != idx ? make_float2(a.x + b.x, a.y - b.y) : make_float2(a.x, 0.f);
    return mir != idx ? make_float2(a.y + b.y, b.x - a.x) : make_float2(a.y, 0.f);
}

// The three component values a half-set point spreads.
__device__ __forceinline__ void half_point_combine(float2 a, float2 b, long long p, long long idx, long long S,
                                                   const Geo &g, int paired, float2 vc[3]) {
    const float2 v = half_point_value(a, b, p, idx, S, paired);
    vc[0] = cscale(v, (float)g.d0);
    vc[1] = cscale(v, (float)g.d1);
    vc[2] = cscale(v, (float)g.d2);
}

// The interpolated value of a half-set point and its mirror: s = sum_i d_i c_i
// at q, conj(s) at -q; at q = 0 (its own mirror) the transform of a real
// volume is real.
__device__ __forceinline__ void store_half_point(float2 *__restrict__ c, long long p, long long idx, long long S,
                                                 const Geo &g, const float2 acc[3]) {
    const float d0 = (float)g.d0, d1 = (float)g.d1, d2 = (float)g.d2;
    float2 s;
    s.x = d0 * acc[0].x + d1 * acc[1].x + d2 * acc[2].x;
    s.y = d0 * acc[0].y + d1 * acc[1].y + d2 * acc[2].y;
    const long long mir = S - 1 - idx;
    if (mir == idx) s.y = 0.f;
    c[p * S + idx] = s;
    if (mir != idx) c[p * S + mir] = cconj(s);
}

}  // namespace lam
