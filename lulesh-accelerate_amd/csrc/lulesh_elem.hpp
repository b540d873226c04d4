// lulesh_elem.hpp -- element-local LULESH arithmetic for gfx950.
//
// Each function evaluates one hexahedral element and keeps, expression by
// expression, the operand order and association of the reference C code it
// cites.  With FMA contraction off (the build passes -ffp-contract=off and
// the pragma below repeats it) every value is then rounded exactly as the
// reference rounds it on the host: the GPU step is bit-identical to the
// reference except for the cube root of the hourglass coefficient, which is
// the project cube root of lulesh_cbrt.h.
#pragma once

#include <hip/hip_runtime.h>

// The mixed-precision translation unit defines LULESH_MIXED_TU and the
// fused float64 build LULESH_FUSED: their results are not bit-matched, so
// there the element templates may fuse multiply-adds.  Everywhere else
// contraction stays off.
#if defined(LULESH_MIXED_TU) || defined(LULESH_FUSED)
#pragma clang fp contract(fast)
#else
#pragma clang fp contract(off)
#endif

#define LULESH_FN static __device__ __forceinline__
// A double constant placed in scalar registers where it is used: the empty
// asm cannot be moved out of a loop, so the constant is not hoisted into
// vector registers that would stay live across the loop.
static __device__ __forceinline__ double lulesh_sconst(double c)
{
    asm volatile("" : "+s"(c));
    return c;
}
#define LULESH_CONST(c) lulesh_sconst(c)
#include "lulesh_cbrt.h"

namespace lulesh {

// Element face boundary-condition bits (reference/C/LULESH-OMP.cc:532-554).
// On the structured cube they follow from the element's (i, j, k): the
// x = 0, y = 0, z = 0 faces are symmetry planes, the far faces free surfaces.

// The geometric helpers are templates on the arithmetic type T: the FP64
// step instantiates them with double (every constant T(c) is then the
// reference's double constant, so the rounding is unchanged), the
// mixed-precision step with float on element-local coordinates.

// 1 / b and a / b in the element arithmetic.  The bit-identical build
// divides, correctly rounded, as the reference does.  The fused build, held
// to the reference's tolerances rather than to its bits, multiplies by the
// hardware reciprocal estimate (relative error below 2^-23) with one
// third-order step (b finite, normal and nonzero): four instructions where
// the divide sequence takes ten.  In
// float (the mixed-precision step) these are plain divides.
__device__ __forceinline__ double elem_recip(double b)
{
#ifdef LULESH_FUSED
    const double r = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
#else
    return 1.0 / b;
#endif
}
__device__ __forceinline__ double elem_quot(double a, double b)
{
#ifdef LULESH_FUSED
    return a * elem_recip(b);
#else
    return a / b;
#endif
}
__device__ __forceinline__ float elem_quot(float a, float b) { return a / b; }

// a / cbrt(d), d > 0 and normal, the hourglass coefficient, in two steps
// with the root first (as the reference orders it): hg_root(d), then
// hg_over_root(a, root).  The bit-identical build takes the project cube
// root (lulesh_cbrt.h) and divides by it.  The fused build takes the
// reciprocal cube root and multiplies by it: the project root's start
// (d = t 2^(3q), t in [1, 8), the cubic fit of t^(-1/3)) and three of its
// Newton steps z <- z + z (1 - t z^3) / 3 (relative error 2.6e-4 ->
// 1.3e-7 -> 3.4e-14 -> rounding), then z 2^-q through the exponent field:
// no root refinement and no divide.
__device__ __forceinline__ double hg_root(double d)
{
#ifdef LULESH_FUSED
    const uint64_t b = __double_as_longlong(d);
    const int e = int((b >> 52) & 0x7ffu) - 1023;
    const int q = int(unsigned(e + 1026) / 3u) - 342;  // floor(e / 3)
    const int r = e - 3 * q;
    const uint64_t frac = b & 0x000fffffffffffffull;
    const double m = __longlong_as_double(frac | (1023ull << 52));
    const double t = __longlong_as_double(frac | (uint64_t(1023 + r) << 52));
    const double third = LULESH_CONST(0.3333333333333333);
    double z = __builtin_fma(m, __builtin_fma(m, __builtin_fma(m, LULESH_CONST(-0.04993701447458462),
                                                               LULESH_CONST(0.3177574893441185)),
                                              LULESH_CONST(-0.809960645949834)),
                             LULESH_CONST(1.5418870676993346));
    const double zc = z * ((r == 1) ? LULESH_CONST(0.7937005259840998)
                                    : LULESH_CONST(0.6299605249474366));
    z = (r == 0) ? z : zc;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double dz = __builtin_fma(-t, (z * z) * z, 1.0);
        z = __builtin_fma(z * dz, third, z);
    }
    return __longlong_as_double(__double_as_longlong(z) - (int64_t(q) << 52));
#else
    return lulesh_cbrt(d);
#endif
}
__device__ __forceinline__ double hg_over_root(double a, double root)
{
#ifdef LULESH_FUSED
    return a * root;
#else
    return a / root;
#endif
}
__device__ __forceinline__ double elem_over_cbrt(double a, double d)
{
    const double root = hg_root(d);
    return hg_over_root(a, root);
}

// fast square root of the arithmetic type: IEEE sqrt in double, the
// hardware v_sqrt_f32 (1 ulp) in float
__device__ __forceinline__ double elem_sqrt(double v) { return sqrt(v); }
__device__ __forceinline__ float elem_sqrt(float v) { return __builtin_amdgcn_sqrtf(v); }

// reference/C/LULESH-OMP.cc:620-706, the Jacobian determinant only (the
// shape-function derivatives of the stress integration are overwritten by
// the node normals before use, :884-888)
template <typename T>
__device__ __forceinline__ T jacobian_volume(const T *x, const T *y, const T *z)
{
    const T e = T(.125);
    const T fjxxi = e * ((x[6] - x[0]) + (x[5] - x[3]) - (x[7] - x[1]) - (x[4] - x[2]));
    const T fjxet = e * ((x[6] - x[0]) - (x[5] - x[3]) + (x[7] - x[1]) - (x[4] - x[2]));
    const T fjxze = e * ((x[6] - x[0]) + (x[5] - x[3]) + (x[7] - x[1]) + (x[4] - x[2]));
    const T fjyxi = e * ((y[6] - y[0]) + (y[5] - y[3]) - (y[7] - y[1]) - (y[4] - y[2]));
    const T fjyet = e * ((y[6] - y[0]) - (y[5] - y[3]) + (y[7] - y[1]) - (y[4] - y[2]));
    const T fjyze = e * ((y[6] - y[0]) + (y[5] - y[3]) + (y[7] - y[1]) + (y[4] - y[2]));
    const T fjzxi = e * ((z[6] - z[0]) + (z[5] - z[3]) - (z[7] - z[1]) - (z[4] - z[2]));
    const T fjzet = e * ((z[6] - z[0]) - (z[5] - z[3]) + (z[7] - z[1]) - (z[4] - z[2]));
    const T fjzze = e * ((z[6] - z[0]) + (z[5] - z[3]) + (z[7] - z[1]) + (z[4] - z[2]));
    const T cjxet = -(fjyxi * fjzze) + (fjzxi * fjyze);
    const T cjyet = (fjxxi * fjzze) - (fjzxi * fjxze);
    const T cjzet = -(fjxxi * fjyze) + (fjyxi * fjxze);
    return T(8.) * (fjxet * cjxet + fjyet * cjyet + fjzet * cjzet);
}

// reference/C/LULESH-OMP.cc:620-706 in full: B[3][4] for nodes 0..3 (nodes
// 4..7 are their negatives in the order 2,3,0,1) and the determinant
template <typename T>
__device__ __forceinline__ T shape_derivatives(const T *x, const T *y, const T *z,
                                               T b[3][4])
{
    const T e = T(.125);
    const T fjxxi = e * ((x[6] - x[0]) + (x[5] - x[3]) - (x[7] - x[1]) - (x[4] - x[2]));
    const T fjxet = e * ((x[6] - x[0]) - (x[5] - x[3]) + (x[7] - x[1]) - (x[4] - x[2]));
    const T fjxze = e * ((x[6] - x[0]) + (x[5] - x[3]) + (x[7] - x[1]) + (x[4] - x[2]));
    const T fjyxi = e * ((y[6] - y[0]) + (y[5] - y[3]) - (y[7] - y[1]) - (y[4] - y[2]));
    const T fjyet = e * ((y[6] - y[0]) - (y[5] - y[3]) + (y[7] - y[1]) - (y[4] - y[2]));
    const T fjyze = e * ((y[6] - y[0]) + (y[5] - y[3]) + (y[7] - y[1]) + (y[4] - y[2]));
    const T fjzxi = e * ((z[6] - z[0]) + (z[5] - z[3]) - (z[7] - z[1]) - (z[4] - z[2]));
    const T fjzet = e * ((z[6] - z[0]) - (z[5] - z[3]) + (z[7] - z[1]) - (z[4] - z[2]));
    const T fjzze = e * ((z[6] - z[0]) + (z[5] - z[3]) + (z[7] - z[1]) + (z[4] - z[2]));

    const T cjxxi = (fjyet * fjzze) - (fjzet * fjyze);
    const T cjxet = -(fjyxi * fjzze) + (fjzxi * fjyze);
    const T cjxze = (fjyxi * fjzet) - (fjzxi * fjyet);
    const T cjyxi = -(fjxet * fjzze) + (fjzet * fjxze);
    const T cjyet = (fjxxi * fjzze) - (fjzxi * fjxze);
    const T cjyze = -(fjxxi * fjzet) + (fjzxi * fjxet);
    const T cjzxi = (fjxet * fjyze) - (fjyet * fjxze);
    const T cjzet = -(fjxxi * fjyze) + (fjyxi * fjxze);
    const T cjzze = (fjxxi * fjyet) - (fjyxi * fjxet);

    b[0][0] = -cjxxi - cjxet - cjxze;
    b[0][1] = cjxxi - cjxet - cjxze;
    b[0][2] = cjxxi + cjxet - cjxze;
    b[0][3] = -cjxxi + cjxet - cjxze;
    b[1][0] = -cjyxi - cjyet - cjyze;
    b[1][1] = cjyxi - cjyet - cjyze;
    b[1][2] = cjyxi + cjyet - cjyze;
    b[1][3] = -cjyxi + cjyet - cjyze;
    b[2][0] = -cjzxi - cjzet - cjzze;
    b[2][1] = cjzxi - cjzet - cjzze;
    b[2][2] = cjzxi + cjzet - cjzze;
    b[2][3] = -cjzxi + cjzet - cjzze;
    return T(8.) * (fjxet * cjxet + fjyet * cjyet + fjzet * cjzet);
}

// reference/C/LULESH-OMP.cc:709-742
template <typename T>
__device__ __forceinline__ void face_normal(T *pfx, T *pfy, T *pfz, const T *x,
                                            const T *y, const T *z, int n0, int n1,
                                            int n2, int n3)
{
    const T h = T(0.5), q = T(0.25);
    const T bx0 = h * (x[n3] + x[n2] - x[n1] - x[n0]);
    const T by0 = h * (y[n3] + y[n2] - y[n1] - y[n0]);
    const T bz0 = h * (z[n3] + z[n2] - z[n1] - z[n0]);
    const T bx1 = h * (x[n2] + x[n1] - x[n3] - x[n0]);
    const T by1 = h * (y[n2] + y[n1] - y[n3] - y[n0]);
    const T bz1 = h * (z[n2] + z[n1] - z[n3] - z[n0]);
    const T ax = q * (by0 * bz1 - bz0 * by1);
    const T ay = q * (bz0 * bx1 - bx0 * bz1);
    const T az = q * (bx0 * by1 - by0 * bx1);
    pfx[n0] += ax; pfx[n1] += ax; pfx[n2] += ax; pfx[n3] += ax;
    pfy[n0] += ay; pfy[n1] += ay; pfy[n2] += ay; pfy[n3] += ay;
    pfz[n0] += az; pfz[n1] += az; pfz[n2] += az; pfz[n3] += az;
}

// reference/C/LULESH-OMP.cc:745-799
template <typename T>
__device__ __forceinline__ void node_normals(T *pfx, T *pfy, T *pfz, const T *x,
                                             const T *y, const T *z)
{
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        pfx[i] = T(0.0);
        pfy[i] = T(0.0);
        pfz[i] = T(0.0);
    }
    face_normal(pfx, pfy, pfz, x, y, z, 0, 1, 2, 3);
    face_normal(pfx, pfy, pfz, x, y, z, 0, 4, 5, 1);
    face_normal(pfx, pfy, pfz, x, y, z, 1, 5, 6, 2);
    face_normal(pfx, pfy, pfz, x, y, z, 2, 6, 7, 3);
    face_normal(pfx, pfy, pfz, x, y, z, 3, 7, 4, 0);
    face_normal(pfx, pfy, pfz, x, y, z, 4, 7, 6, 5);
}

// reference/C/LULESH-OMP.cc:979-1006; the node-by-node argument lists of
// CalcElemVolumeDerivative are :1008-1048
template <typename T>
__device__ __forceinline__ void volu_der(const T *x, const T *y, const T *z, int a0,
                                         int a1, int a2, int a3, int a4, int a5,
                                         T &dvdx, T &dvdy, T &dvdz)
{
    const T twelfth = T(1.0 / 12.0);
    const T x0 = x[a0], x1 = x[a1], x2 = x[a2], x3 = x[a3], x4 = x[a4], x5 = x[a5];
    const T y0 = y[a0], y1 = y[a1], y2 = y[a2], y3 = y[a3], y4 = y[a4], y5 = y[a5];
    const T z0 = z[a0], z1 = z[a1], z2 = z[a2], z3 = z[a3], z4 = z[a4], z5 = z[a5];
    dvdx = (y1 + y2) * (z0 + z1) - (y0 + y1) * (z1 + z2) +
           (y0 + y4) * (z3 + z4) - (y3 + y4) * (z0 + z4) -
           (y2 + y5) * (z3 + z5) + (y3 + y5) * (z2 + z5);
    dvdy = -(x1 + x2) * (z0 + z1) + (x0 + x1) * (z1 + z2) -
           (x0 + x4) * (z3 + z4) + (x3 + x4) * (z0 + z4) +
           (x2 + x5) * (z3 + z5) - (x3 + x5) * (z2 + z5);
    dvdz = -(y1 + y2) * (x0 + x1) + (y0 + y1) * (x1 + x2) -
           (y0 + y4) * (x3 + x4) + (y3 + y4) * (x0 + x4) +
           (y2 + y5) * (x3 + x5) - (y3 + y5) * (x2 + x5);
    dvdx *= twelfth;
    dvdy *= twelfth;
    dvdz *= twelfth;
}

// Flanagan-Belytschko hourglass base vectors (reference/C/LULESH-OMP.cc:
// 1252-1285), one row per mode, entries +-1
template <typename T = double>
__device__ __forceinline__ T fb_gamma(int mode, int node)
{
    constexpr signed char g[4][8] = {
        {1, 1, -1, -1, -1, -1, 1, 1},
        {1, -1, -1, 1, -1, 1, 1, -1},
        {1, -1, 1, -1, 1, -1, 1, -1},
        {-1, 1, -1, 1, 1, -1, 1, -1},
    };
    return T(g[mode][node]);
}

// reference/C/LULESH-OMP.cc:1706-1789
template <typename T>
__device__ __forceinline__ T triple_product(T x1, T y1, T z1, T x2, T y2, T z2, T x3,
                                            T y3, T z3)
{
    return x1 * (y2 * z3 - z2 * y3) + x2 * (z1 * y3 - y1 * z3) +
           x3 * (y1 * z2 - z1 * y2);
}

template <typename T>
__device__ __forceinline__ T elem_volume(const T *x, const T *y, const T *z)
{
    const T twelveth = T(1.0 / 12.0);
    const T dx61 = x[6] - x[1], dy61 = y[6] - y[1], dz61 = z[6] - z[1];
    const T dx70 = x[7] - x[0], dy70 = y[7] - y[0], dz70 = z[7] - z[0];
    const T dx63 = x[6] - x[3], dy63 = y[6] - y[3], dz63 = z[6] - z[3];
    const T dx20 = x[2] - x[0], dy20 = y[2] - y[0], dz20 = z[2] - z[0];
    const T dx50 = x[5] - x[0], dy50 = y[5] - y[0], dz50 = z[5] - z[0];
    const T dx64 = x[6] - x[4], dy64 = y[6] - y[4], dz64 = z[6] - z[4];
    const T dx31 = x[3] - x[1], dy31 = y[3] - y[1], dz31 = z[3] - z[1];
    const T dx72 = x[7] - x[2], dy72 = y[7] - y[2], dz72 = z[7] - z[2];
    const T dx43 = x[4] - x[3], dy43 = y[4] - y[3], dz43 = z[4] - z[3];
    const T dx57 = x[5] - x[7], dy57 = y[5] - y[7], dz57 = z[5] - z[7];
    const T dx14 = x[1] - x[4], dy14 = y[1] - y[4], dz14 = z[1] - z[4];
    const T dx25 = x[2] - x[5], dy25 = y[2] - y[5], dz25 = z[2] - z[5];
    T volume =
        triple_product(dx31 + dx72, dx63, dx20, dy31 + dy72, dy63, dy20,
                       dz31 + dz72, dz63, dz20) +
        triple_product(dx43 + dx57, dx64, dx70, dy43 + dy57, dy64, dy70,
                       dz43 + dz57, dz64, dz70) +
        triple_product(dx14 + dx25, dx61, dx50, dy14 + dy25, dy61, dy50,
                       dz14 + dz25, dz61, dz50);
    volume *= twelveth;
    return volume;
}

// reference/C/LULESH-OMP.cc:1799-1819
template <typename T>
__device__ __forceinline__ T area_face(const T *x, const T *y, const T *z, int n0,
                                       int n1, int n2, int n3)
{
    const T fx = (x[n2] - x[n0]) - (x[n3] - x[n1]);
    const T fy = (y[n2] - y[n0]) - (y[n3] - y[n1]);
    const T fz = (z[n2] - z[n0]) - (z[n3] - z[n1]);
    const T gx = (x[n2] - x[n0]) + (x[n3] - x[n1]);
    const T gy = (y[n2] - y[n0]) + (y[n3] - y[n1]);
    const T gz = (z[n2] - z[n0]) + (z[n3] - z[n1]);
    return (fx * fx + fy * fy + fz * fz) * (gx * gx + gy * gy + gz * gz) -
           (fx * gx + fy * gy + fz * gz) * (fx * gx + fy * gy + fz * gz);
}

// std::max(a, b) as the reference's libstdc++ evaluates it
template <typename T>
__device__ __forceinline__ T ref_max(T a, T b)
{
    return (a < b) ? b : a;
}

// reference/C/LULESH-OMP.cc:1821-1862
template <typename T>
__device__ __forceinline__ T characteristic_length(const T *x, const T *y, const T *z,
                                                   T volume)
{
    T cl = T(0.0);
    cl = ref_max(area_face(x, y, z, 0, 1, 2, 3), cl);
    cl = ref_max(area_face(x, y, z, 4, 5, 6, 7), cl);
    cl = ref_max(area_face(x, y, z, 0, 1, 5, 4), cl);
    cl = ref_max(area_face(x, y, z, 1, 2, 6, 5), cl);
    cl = ref_max(area_face(x, y, z, 2, 3, 7, 6), cl);
    cl = ref_max(area_face(x, y, z, 3, 0, 4, 7), cl);
    return elem_quot(T(4.0) * volume, elem_sqrt(cl));
}

// Equation of state of one element: CalcEnergyForElems with its three
// CalcPressureForElems evaluations and CalcSoundSpeedForElems
// (reference/C/LULESH-OMP.cc:2384-2561; lulesh-2.0.3/lulesh.cc:2043-2231).
struct EosConst {
    double e_cut, p_cut, q_cut, eosvmax, eosvmin, pmin, emin, rho0;
    double ss_tiny, ss_floor;
    bool unit_rho0;  // rho0 == 1: x / rho0 is x exactly (see eos_element)
};

struct EosOut {
    double p, e, q, ss;
};

// Correctly rounded square root of s >= 2^-767 (and of +inf and NaN): the
// Newton-Raphson refinement of the hardware reciprocal square root that the
// compiler emits for sqrt(double) on gfx950 (two coupled iterations on the
// root g*s and the half-reciprocal g/2, then two residual corrections
// d = s - r*r, r += d*h), without the input scaling it adds for inputs
// below 2^-767 and without its zero test.  For such s it is sqrt(s) bit for
// bit (checked against the host's sqrt in the tests); the EOS calls it only
// above its sound-speed floor (>= 1e-37).
__device__ __forceinline__ double sqrt_above_tiny(double s)
{
    const double g = __builtin_amdgcn_rsq(s);
    double r = s * g;
    double h = g * 0.5;
    const double e = __builtin_fma(-h, r, 0.5);
    r = __builtin_fma(r, e, r);
    h = __builtin_fma(h, e, h);
    double d = __builtin_fma(-r, r, s);
    r = __builtin_fma(d, h, r);
    d = __builtin_fma(-r, r, s);
    r = __builtin_fma(d, h, r);
    return (s == __builtin_inf()) ? s : r;
}

#ifdef LULESH_FUSED
// sqrt_above_tiny without its second residual correction: the error before the
// last rounding, the square of the estimate's after one iteration, is about
// 2^-94 of the root, so the last bit is another one only where the root lies
// that near to the middle between two doubles.  Of 2e5 sound speeds none
// was (the tests).
__device__ __forceinline__ double root_above_tiny(double s)
{
    const double g = __builtin_amdgcn_rsq(s);
    double r = s * g;
    double h = g * 0.5;
    const double e = __builtin_fma(-h, r, 0.5);
    r = __builtin_fma(r, e, r);
    h = __builtin_fma(h, e, h);
    r = __builtin_fma(__builtin_fma(-r, r, s), h, r);
    return (s == __builtin_inf()) ? s : r;
}
#endif

// the sound speed squared over rho0; UnitRho0 (rho0 == 1, where x / rho0
// is x exactly) leaves the divide out at compile time
template <bool UnitRho0>
__device__ __forceinline__ double eos_sound(double pbvc, double e, double vv,
                                            double bvc, double p, double rho0,
                                            double tiny, double floor_v)
{
    double s = (pbvc * e + vv * bvc * p);
    if (!UnitRho0) {
        s = s / rho0;
    }
    if (s <= tiny) {
        s = floor_v;
    } else {
        s = sqrt_above_tiny(s);
    }
    return s;
}

__device__ __forceinline__ double eos_pressure(double bvc, double e,
                                               double vnewc, const EosConst &c)
{
    double p = bvc * e;
    if (fabs(p) < c.p_cut) p = 0.0;
    if (vnewc >= c.eosvmax) p = 0.0;
    if (p < c.pmin) p = c.pmin;
    return p;
}

// UnitRho0 must equal c.unit_rho0: the caller picks the instance, so the
// unit-density case carries no divides by rho0 and no selects between the
// two results
#ifdef LULESH_FUSED
// The fused build works with the reciprocal volumes 1 / v and 1 / vhalf
// themselves, where the reference adds 1 to compressions formed by
// subtracting it, and so needs neither a reciprocal for vhalf nor the
// products vhalf^2 (1 / vhalf) and v^2 (1 / v) of the sound speeds: an
// evaluation is 159 vector instructions, 211 in the reference's form.
template <bool UnitRho0>
__device__ __forceinline__ EosOut eos_element(double vnewc, double e_old,
                                              double delvc, double p_old,
                                              double q_old, double qq_old,
                                              double ql_old, const EosConst &c)
{
    const double c1s = 2.0 / 3.0;
    double vhalf = vnewc - delvc * .5;
    double r = elem_recip(vnewc), r_half = elem_recip(vhalf);
    double v2r = vnewc;  // vnewc^2 r
    if (c.eosvmin != 0.) {
        if (vnewc <= c.eosvmin) {
            vhalf = vnewc;
            r_half = r;
        }
    }
    if (c.eosvmax != 0.) {
        if (vnewc >= c.eosvmax) {  // the compressions are 0
            p_old = 0.;
            r = 1.;
            r_half = 1.;
            vhalf = 1.;
            v2r = vnewc * vnewc;
        }
    }
    const double bvc_half = c1s * r_half, bvc = c1s * r;
    const double pq_old = p_old + q_old;
    double e_new = __builtin_fma(-0.5 * delvc, pq_old, e_old);
    if (e_new < c.emin) e_new = c.emin;
    const double p_half = eos_pressure(bvc_half, e_new, vnewc, c);
    const bool expanding = delvc > 0.;
    // c1s e + v^2 bvc p, the sound speed squared times rho0
    auto sound = [&](double v, double e, double p) {
        double s = c1s * __builtin_fma(v, p, e);
        if (!UnitRho0) {
            s = s / c.rho0;
        }
        return (s <= c.ss_tiny) ? c.ss_floor : root_above_tiny(s);
    };
    double q_new = 0.;
    if (!expanding) {
        q_new = __builtin_fma(sound(vhalf, e_new, p_half), ql_old, qq_old);
    }
    const double pq_half = p_half + q_new;
    e_new = __builtin_fma(0.5 * delvc, __builtin_fma(3.0, pq_old, -4.0 * pq_half), e_new);
    if (fabs(e_new) < c.e_cut) e_new = 0.;
    if (e_new < c.emin) e_new = c.emin;
    double p_new = eos_pressure(bvc, e_new, vnewc, c);
    double q_tilde = 0.;
    if (!expanding) {
        q_tilde = __builtin_fma(sound(v2r, e_new, p_new), ql_old, qq_old);
    }
    const double sum = __builtin_fma(7.0, pq_old, __builtin_fma(-8.0, pq_half, p_new + q_tilde));
    e_new = __builtin_fma(-sum, delvc * (1.0 / 6.0), e_new);
    if (fabs(e_new) < c.e_cut) e_new = 0.;
    if (e_new < c.emin) e_new = c.emin;
    p_new = eos_pressure(bvc, e_new, vnewc, c);
    EosOut o;
    o.ss = sound(v2r, e_new, p_new);
    if (delvc <= 0.) {
        q_new = __builtin_fma(o.ss, ql_old, qq_old);
        if (fabs(q_new) < c.q_cut) q_new = 0.;
    }
    o.p = p_new;
    o.e = e_new;
    o.q = q_new;
    return o;
}
#else
template <bool UnitRho0>
__device__ __forceinline__ EosOut eos_element(double vnewc, double e_old,
                                              double delvc, double p_old,
                                              double q_old, double qq_old,
                                              double ql_old, const EosConst &c)
{
    const double c1s = 2.0 / 3.0;
    const double work = 0.;
    double compression = elem_recip(vnewc) - 1.;
    const double vchalf = vnewc - delvc * .5;
    double comp_half_step = elem_recip(vchalf) - 1.;
    if (c.eosvmin != 0.) {
        if (vnewc <= c.eosvmin) comp_half_step = compression;
    }
    if (c.eosvmax != 0.) {
        if (vnewc >= c.eosvmax) {
            p_old = 0.;
            compression = 0.;
            comp_half_step = 0.;
        }
    }
    double e_new = e_old - 0.5 * delvc * (p_old + q_old) + 0.5 * work;
    if (e_new < c.emin) e_new = c.emin;

    double bvc = c1s * (comp_half_step + 1.);
    double pbvc = c1s;
    const double p_half_step = eos_pressure(bvc, e_new, vnewc, c);

    const double vhalf = elem_recip(1. + comp_half_step);
    double q_new;
    if (delvc > 0.) {
        q_new = 0.;
    } else {
        const double ssc = eos_sound<UnitRho0>(pbvc, e_new, vhalf * vhalf, bvc, p_half_step,
                                               c.rho0, c.ss_tiny, c.ss_floor);
        q_new = (ssc * ql_old + qq_old);
    }
    e_new = e_new + 0.5 * delvc * (3.0 * (p_old + q_old) - 4.0 * (p_half_step + q_new));
    e_new += 0.5 * work;
    if (fabs(e_new) < c.e_cut) e_new = 0.;
    if (e_new < c.emin) e_new = c.emin;

    bvc = c1s * (compression + 1.);
    pbvc = c1s;
    double p_new = eos_pressure(bvc, e_new, vnewc, c);
    {
        const double sixth = 1.0 / 6.0;
        double q_tilde;
        if (delvc > 0.) {
            q_tilde = 0.;
        } else {
            const double ssc = eos_sound<UnitRho0>(pbvc, e_new, vnewc * vnewc, bvc, p_new,
                                                   c.rho0, c.ss_tiny, c.ss_floor);
            q_tilde = (ssc * ql_old + qq_old);
        }
        e_new = e_new - (7.0 * (p_old + q_old) - 8.0 * (p_half_step + q_new) +
                         (p_new + q_tilde)) * delvc * sixth;
        if (fabs(e_new) < c.e_cut) e_new = 0.;
        if (e_new < c.emin) e_new = c.emin;
    }
    bvc = c1s * (compression + 1.);
    pbvc = c1s;
    p_new = eos_pressure(bvc, e_new, vnewc, c);
    // the sound speed of the last q and of the time constraint (CalcQForElems
    // and CalcSoundSpeedForElems) are the same expression
    EosOut o;
    o.ss = eos_sound<UnitRho0>(pbvc, e_new, vnewc * vnewc, bvc, p_new, c.rho0, c.ss_tiny,
                               c.ss_floor);
    if (delvc <= 0.) {
        q_new = (o.ss * ql_old + qq_old);
        if (fabs(q_new) < c.q_cut) q_new = 0.;
    }
    o.p = p_new;
    o.e = e_new;
    o.q = q_new;
    return o;
}
#endif  // LULESH_FUSED

}  // namespace lulesh
