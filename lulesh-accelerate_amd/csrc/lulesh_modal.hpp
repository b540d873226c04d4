// lulesh_modal.hpp -- a hexahedron's forces in terms of its modes.
//
// Used where results are held to the reference's tolerances rather than to
// its bits.  The eight corner values of a field are replaced by their sums
// with the signs of xi, eta, zeta, eta*zeta, zeta*xi, xi*eta and
// xi*eta*zeta (the sum without signs never enters):
//
//   A1 A2 A3   the directions (8 times the Jacobian's columns at the centre)
//   H1 H2 H3   the bilinear modes, H4 the trilinear one; the last four are
//              the Flanagan-Belytschko base vectors (reference/C/
//              LULESH-OMP.cc:1252-1285) applied to the coordinates
//
// In these, with C1 = A2 x A3, D1 = H3 x H2 and their cyclic forms,
//   volume          512 V = A1.C1 + (H3.(A2 x H1) + H2.(H1 x A3) + A1.(H3 x H2)) / 3
//   corner normals  64 n_c = s1 (C1+D1) + s2 (C2+D2) + s3 (C3+D3)
//                   (the quarter sums of the face normals, :745-799: of the
//                   seven modes only three are non-zero)
//   dV/dx_c         sum over the six modes of sign_k(c) g_k / 64, with
//                   3 g_A1 = 3 C1 + D1, 3 g_H1 = H3 x A2 + A3 x H2, cyclic
//                   (:979-1048; H4 does not change the volume)
// so the hourglass force (:1326-1473), a product of 8 x 4 matrices per
// component in corner values, becomes one with the 6 x 4 matrix
// M_ik = g_k . H_i / V and the velocities' modes.  An element's stress and
// hourglass forces take about 500 instructions this way, against about 1100
// corner by corner.
//
// Every difference of coordinates is taken before any sum, between corners
// one edge apart: it is exact or nearly so, and the modes carry no more
// rounding than the corner forms.
#pragma once

#include "lulesh_elem.hpp"

// Every multiply-add is written out: two kernels that share a function get the
// same bits from it whatever they inline it into.
#pragma clang fp contract(off)

namespace lulesh {

template <typename T>
struct Vec3 {
    T x, y, z;
};

template <typename T>
__device__ __forceinline__ T fused_madd(T a, T b, T c);
template <>
__device__ __forceinline__ double fused_madd(double a, double b, double c)
{
    return __builtin_fma(a, b, c);
}
template <>
__device__ __forceinline__ float fused_madd(float a, float b, float c)
{
    return __builtin_fmaf(a, b, c);
}

template <typename T>
__device__ __forceinline__ Vec3<T> cross(const Vec3<T> &a, const Vec3<T> &b)
{
    return {fused_madd(a.y, b.z, -(a.z * b.y)), fused_madd(a.z, b.x, -(a.x * b.z)),
            fused_madd(a.x, b.y, -(a.y * b.x))};
}
// a x b + c
template <typename T>
__device__ __forceinline__ Vec3<T> cross_add(const Vec3<T> &a, const Vec3<T> &b, const Vec3<T> &c)
{
    return {fused_madd(a.y, b.z, fused_madd(-a.z, b.y, c.x)),
            fused_madd(a.z, b.x, fused_madd(-a.x, b.z, c.y)),
            fused_madd(a.x, b.y, fused_madd(-a.y, b.x, c.z))};
}
// rounded alike in x and y
template <typename T>
__device__ __forceinline__ T dot(const Vec3<T> &a, const Vec3<T> &b)
{
    return fused_madd(a.z, b.z, a.x * b.x + a.y * b.y);
}
// one instruction less
template <typename T>
__device__ __forceinline__ T dot_xyz(const Vec3<T> &a, const Vec3<T> &b)
{
    return fused_madd(a.z, b.z, fused_madd(a.y, b.y, a.x * b.x));
}
template <typename T>
__device__ __forceinline__ Vec3<T> scale(T s, const Vec3<T> &a)
{
    return {s * a.x, s * a.y, s * a.z};
}

// The four corner values of a face of constant zeta (corner 0, and 1, 2, 3
// counter-clockwise), as corner 0, the sum of the others' differences from
// it, and the face's xi, eta and xi*eta modes.
template <typename T>
struct FaceModes {
    T v0, rest, xi, eta, xieta;
};

template <typename T>
__device__ __forceinline__ FaceModes<T> face_modes(T v0, T v1, T v2, T v3)
{
    const T e = v1 - v0, f = v2 - v3, g = v3 - v0;
    FaceModes<T> m;
    m.v0 = v0;
    m.xi = e + f;
    m.xieta = f - e;
    m.eta = fused_madd(T(2), g, m.xieta);   // (v3 - v0) + (v2 - v1)
    m.rest = fused_madd(T(2), g, m.xi);     // (v1 - v0) + (v2 - v0) + (v3 - v0)
    return m;
}

// the element's modes of one field from its low and high face
template <typename T>
struct ElemModes {
    T a1, a2, a3, h1, h2, h3, h4;
};

template <typename T>
__device__ __forceinline__ ElemModes<T> elem_modes(const FaceModes<T> &lo, const FaceModes<T> &hi)
{
    ElemModes<T> m;
    m.a1 = hi.xi + lo.xi;
    m.h2 = hi.xi - lo.xi;
    m.a2 = hi.eta + lo.eta;
    m.h1 = hi.eta - lo.eta;
    m.h3 = hi.xieta + lo.xieta;
    m.h4 = hi.xieta - lo.xieta;
    m.a3 = fused_madd(T(4), hi.v0 - lo.v0, hi.rest - lo.rest);
    return m;
}

// 1 / sqrt(s), s > 0 and normal: the hardware estimate (relative error below
// 2^-23) with one third-order step, whose remainder is its cube.
__device__ __forceinline__ double recip_root(double s)
{
    const double g = __builtin_amdgcn_rsq(s);
    const double e = __builtin_fma(-(s * g), g, 1.0);
    return __builtin_fma(g * e, __builtin_fma(e, 0.375, 0.5), g);
}

// The volume from the corners (CalcElemVolume, :1739-1789: three triple
// products of diagonals).  The modes would give it in 50 instructions less;
// but a rounding of the volume is one of the energy in every cycle, what
// asymmetry a run of the symmetric blast shows is that rounding's, and in
// this form it is the reference's.
__device__ __forceinline__ double corner_volume(const double *x, const double *y, const double *z)
{
    auto diff = [&](int i, int j) {
        return Vec3<double>{x[i] - x[j], y[i] - y[j], z[i] - z[j]};
    };
    auto sum = [](const Vec3<double> &a, const Vec3<double> &b) {
        return Vec3<double>{a.x + b.x, a.y + b.y, a.z + b.z};
    };
    double v = dot(sum(diff(3, 1), diff(7, 2)), cross(diff(6, 3), diff(2, 0)));
    v += dot(sum(diff(4, 3), diff(5, 7)), cross(diff(6, 4), diff(7, 0)));
    v += dot(sum(diff(1, 4), diff(2, 5)), cross(diff(6, 1), diff(5, 0)));
    return v * (1.0 / 12.0);
}

// the modes of a field from its eight corner values
__device__ __forceinline__ ElemModes<double> corner_modes(const double *v)
{
    return elem_modes(face_modes(v[0], v[1], v[2], v[3]), face_modes(v[4], v[5], v[6], v[7]));
}

// The monotonic-Q velocity gradient of direction k (:2034-2180): the cross
// product of the other two directions, dotted with its velocity mode; norm64
// is 1 / (64 (volume + ptiny)).
__device__ __forceinline__ double q_gradient(const Vec3<double> &c, const Vec3<double> &u,
                                             double norm64)
{
    return dot_xyz(c, u) * norm64;
}
__device__ __forceinline__ double q_norm64(double vol)
{
    return elem_recip(vol + 1.e-36) * 0.015625;
}

// Kinematics of one element (:1821-1862, :1927-2032) and its monotonic-Q
// gradients, in two parts so that the corner positions need not be held
// beside the velocities: the shape from the corners xyz[component][corner],
// and the rest from the shape and the velocities' modes.
struct ElemShape {
    double volume;
    double area;     // 16 times the squared area of the largest face, squared
    Vec3<double> a[3];  // the directions
};

__device__ __forceinline__ ElemShape elem_shape(const double (&xyz)[3][8])
{
    ElemShape s;
    s.volume = corner_volume(xyz[0], xyz[1], xyz[2]);
    const ElemModes<double> x = corner_modes(xyz[0]), y = corner_modes(xyz[1]),
                            z = corner_modes(xyz[2]);
    s.a[0] = {x.a1, y.a1, z.a1};
    s.a[1] = {x.a2, y.a2, z.a2};
    s.a[2] = {x.a3, y.a3, z.a3};
    const Vec3<double> h[3] = {{x.h1, y.h1, z.h1}, {x.h2, y.h2, z.h2}, {x.h3, y.h3, z.h3}};
    // the largest of the six faces' |f|^2 |g|^2 - (f.g)^2, f and g twice the
    // face's directions
    s.area = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = (k + 1) % 3, j = (k + 2) % 3;  // the faces of direction k
        const Vec3<double> &f = s.a[i], &g = s.a[j], &hf = h[j], &hg = h[i];
#pragma unroll
        for (int side = -1; side <= 1; side += 2) {
            const Vec3<double> p = {f.x + side * hf.x, f.y + side * hf.y, f.z + side * hf.z};
            const Vec3<double> q = {g.x + side * hg.x, g.y + side * hg.y, g.z + side * hg.z};
            const double pq = dot_xyz(p, q);
            s.area = __builtin_fmax(s.area,
                                    __builtin_fma(dot_xyz(p, p), dot_xyz(q, q), -(pq * pq)));
        }
    }
    return s;
}

// relative volume, characteristic length, rate of volume change, and delv /
// delx of each direction; u[k]: the velocity's modes of direction k
struct ElemKinematics {
    double vnew, arealg, vdov, delv[3], delx[3];
};

__device__ __forceinline__ ElemKinematics elem_kinematics(const ElemShape &s,
                                                          const Vec3<double> (&u)[3],
                                                          double volo, double dt)
{
    ElemKinematics r;
    r.vnew = s.volume * elem_recip(volo);
    r.arealg = 16.0 * s.volume * recip_root(s.area);
    // half-step geometry
    const double dt2 = 0.5 * dt;
    Vec3<double> b[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        b[k] = {__builtin_fma(-dt2, u[k].x, s.a[k].x), __builtin_fma(-dt2, u[k].y, s.a[k].y),
                __builtin_fma(-dt2, u[k].z, s.a[k].z)};
    }
    const Vec3<double> c0 = cross(b[1], b[2]), c1 = cross(b[2], b[0]), c2 = cross(b[0], b[1]);
    r.vdov = (dot_xyz(c0, u[0]) + dot_xyz(c1, u[1]) + dot_xyz(c2, u[2])) *
             elem_recip(dot_xyz(b[2], c2));
    const double vol = volo * r.vnew;
    const double norm64 = q_norm64(vol);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const Vec3<double> c = cross(s.a[(k + 1) % 3], s.a[(k + 2) % 3]);
        r.delv[k] = q_gradient(c, u[k], norm64);
        r.delx[k] = vol * recip_root(__builtin_fma(dot_xyz(c, c), 1.0 / 256.0, 1.e-36));
    }
    return r;
}

// The velocity gradient alone, of direction 0 or 1: the same bits.  a:
// the directions, u: that direction's velocity mode.
__device__ __forceinline__ double elem_gradient(double volume, const Vec3<double> (&a)[3],
                                                const Vec3<double> &u, double volo, bool eta)
{
    const double vol = volo * (volume * elem_recip(volo));
    const Vec3<double> p = eta ? a[2] : a[1], q = eta ? a[0] : a[2];
    return q_gradient(cross(p, q), u, q_norm64(vol));
}

// What the corner forces need of the element's shape: the stress normals
// n[k] (times 64) and the hourglass matrix mat[i][k] (i = H1..H4;
// k = A1..A3, H1..H3); det: 512 times the Jacobian determinant at the centre.
template <typename T>
struct ForceShape {
    Vec3<T> n[3];
    T mat[4][6];
    T det;
};

// volinv: 1 / V
template <typename T>
__device__ __forceinline__ void force_shape(const ElemModes<T> &x, const ElemModes<T> &y,
                                            const ElemModes<T> &z, T volinv,
                                            ForceShape<T> &s)
{
    const Vec3<T> a1 = {x.a1, y.a1, z.a1}, a2 = {x.a2, y.a2, z.a2}, a3 = {x.a3, y.a3, z.a3};
    const Vec3<T> h1 = {x.h1, y.h1, z.h1}, h2 = {x.h2, y.h2, z.h2}, h3 = {x.h3, y.h3, z.h3};
    const Vec3<T> h4 = {x.h4, y.h4, z.h4};
    const Vec3<T> c[3] = {cross(a2, a3), cross(a3, a1), cross(a1, a2)};
    const Vec3<T> d[3] = {cross(h3, h2), cross(h1, h3), cross(h2, h1)};
    s.det = dot_xyz(a1, c[0]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s.n[k] = {c[k].x + d[k].x, c[k].y + d[k].y, c[k].z + d[k].z};
    }
    // 192 g_k (3 x 64), so the H_i carry 1 / (192 V)
    Vec3<T> g[6];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        g[k] = {fused_madd(T(3), c[k].x, d[k].x), fused_madd(T(3), c[k].y, d[k].y),
                fused_madd(T(3), c[k].z, d[k].z)};
    }
    g[3] = cross_add(h3, a2, cross(a3, h2));
    g[4] = cross_add(h1, a3, cross(a1, h3));
    g[5] = cross_add(a2, h1, cross(h2, a1));
    const T vs = volinv * T(1.0 / 192.0);
    const Vec3<T> h[4] = {scale(vs, h1), scale(vs, h2), scale(vs, h3), scale(vs, h4)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            s.mat[i][k] = dot_xyz(h[i], g[k]);
        }
    }
}

// The modes of one component of the element's corner forces: stress
// (press64 n, press64 = (p + q) / 64) and hourglass
// (coef = -hgcoef 0.01 ss m / cbrt(V)) from the component's velocity modes.
// n1, n2, n3: that component of the three stress normals.
template <typename T>
__device__ __forceinline__ ElemModes<T> force_modes(const ForceShape<T> &s, T n1, T n2, T n3,
                                                    T press64, T coef, const ElemModes<T> &u)
{
    const T uk[6] = {u.a1, u.a2, u.a3, u.h1, u.h2, u.h3};
    T w[4] = {u.h1, u.h2, u.h3, u.h4};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            w[i] = fused_madd(-s.mat[i][k], uk[k], w[i]);
        }
        w[i] = coef * w[i];
    }
    T f[6] = {press64 * n1, press64 * n2, press64 * n3, w[0], w[1], w[2]};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            f[k] = fused_madd(-s.mat[i][k], w[i], f[k]);
        }
    }
    return {f[0], f[1], f[2], f[3], f[4], f[5], w[3]};
}

}  // namespace lulesh
