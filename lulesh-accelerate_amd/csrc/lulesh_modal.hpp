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
template <typename T>
__device__ __forceinline__ T dot(const Vec3<T> &a, const Vec3<T> &b)
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
    s.det = dot(a1, c[0]);
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
            s.mat[i][k] = dot(h[i], g[k]);
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
