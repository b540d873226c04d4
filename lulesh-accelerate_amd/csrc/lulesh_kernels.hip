// lulesh_kernels.hip -- the element phases and the time step of a cycle.
//
// Cycle = TimeIncrement + LagrangeLeapFrog (reference/C/LULESH-OMP.cc:
// 3179-3188; lulesh-2.0.3/lulesh.cc:2771-2781).  Kernels, in launch order:
//
//   k_force_sweep      TimeIncrement (:557-604; start_cycle), then
//                      LagrangeNodal: forces, acceleration, boundary
//                      conditions, velocity, position (lulesh_force.hip)
//   k_kinematics_q     per element: kinematics and the monotonic-Q gradients
//                      (:1927-2180)
//   k_q_eos_dt         per element in region order: monotonic-Q limiter
//                      (:2182-2320), qstop check (:2368-2381), EOS with the
//                      region repetitions (:2384-2761; lulesh-2.0.3/lulesh.cc:
//                      2357-2430), volume update (:2763-2782) and the
//                      Courant / hydro minima (:2799-2942), which the last
//                      block to finish applies to dtcourant / dthydro
//
// Every kernel returns at once when the cycle is not active (the run is
// over or an earlier phase raised an error), so whole batches of cycles can
// be queued without a host round trip per cycle.
#include <type_traits>

#include "lulesh_kernels.hpp"

#include "lulesh_elem.hpp"
#ifdef LULESH_FUSED
#include "lulesh_modal.hpp"
#endif
#include "lulesh_mlp.hpp"

// FMA contraction off: every value rounded as the reference rounds it;
// the fused build (LULESH_FUSED) lets multiply-adds fuse
#ifdef LULESH_FUSED
#pragma clang fp contract(fast)
#else
#pragma clang fp contract(off)
#endif

namespace lulesh {
LULESH_VARIANT_BEGIN

namespace {

constexpr double kBig = 1.0e+20;

// a * b + c: two roundings in the bit-identical build, one in the fused
// build.  Where the fused build has to give the same bits from two kernels,
// its multiply-adds are written out like this rather than left to the
// compiler, whose choice depends on what surrounds them (and contraction is
// off where they stand).
__device__ __forceinline__ double madd(double a, double b, double c)
{
#ifdef LULESH_FUSED
    return __builtin_fma(a, b, c);
#else
    return a * b + c;
#endif
}

__device__ __forceinline__ unsigned long long as_bits(double v)
{
    return static_cast<unsigned long long>(__double_as_longlong(v));
}

__device__ __forceinline__ double from_bits(unsigned long long b)
{
    return __longlong_as_double(static_cast<long long>(b));
}

__device__ __forceinline__ void raise_error(DevScalars *s, int code)
{
    // the first error of a cycle wins; later phases see it and return
    atomicCAS(&s->error, 0, code);
}

// a + b of two products, each rounded on its own
__device__ __forceinline__ double add(double a, double b)
{
#pragma clang fp contract(off)
    return a + b;
}

// element (i, j, k) of a flat element index
template <class F>
__device__ __forceinline__ void elem_ijk(const F &f, int el, int &i, int &j,
                                         int &k)
{
    const unsigned q1 = fast_div(unsigned(el), f.div_nx);
    i = el - int(q1) * f.nx;
    const unsigned q2 = fast_div(q1, f.div_nx);
    j = int(q1) - int(q2) * f.nx;
    k = int(q2);
}

}  // namespace

// one thread per member
__global__ void k_time_increment_batch(const BatchMember *__restrict__ members,
                                       const BatchWork *__restrict__ work, int ic_mode)
{
    const int n = work->num_members;
    for (int m = int(threadIdx.x); m < n; m += int(blockDim.x)) {
        DevScalars *const s = members[m].s;
        DevScalars t = *s;  // on a register copy, as in start_cycle
        time_increment(&t, ic_mode);
        *s = t;
    }
}

// ---------------------------------------------------------------------------
// Kinematics (CalcKinematicsForElems + CalcLagrangeElements,
// reference/C/LULESH-OMP.cc:1927-2032) and the monotonic-Q gradients
// (CalcMonotonicQGradientsForElems, :2034-2180) of each element, sharing one
// read of its eight advanced nodes.
// ---------------------------------------------------------------------------
namespace {

// the element's eight nodes are given (structured or from a node list);
// OneTrip: all node loads before any arithmetic (see below)
template <bool OneTrip, class F>
__device__ __forceinline__ void kinematics_q_nodes(const F &f, DevScalars *s,
                                                   int el, const int (&nodes)[8])
{
    // the loop scalars are read through a global pointer: scalar loads
    const LULESH_AS_GLOBAL DevScalars *gs = (const LULESH_AS_GLOBAL DevScalars *)s;
    const int par = wave_uniform(gs->cur);
    const double dt = wave_uniform(gs->deltatime);
    typename F::CPtr __restrict__ px = parity_copy(f.x, par);
    typename F::CPtr __restrict__ py = parity_copy(f.y, par);
    typename F::CPtr __restrict__ pz = parity_copy(f.z, par);
    typename F::CPtr __restrict__ pxd = parity_copy(f.xd, par);
    typename F::CPtr __restrict__ pyd = parity_copy(f.yd, par);
    typename F::CPtr __restrict__ pzd = parity_copy(f.zd, par);
    double xyz[3][8], xv[8], yv[8], zv[8];
    double(&x)[8] = xyz[0], (&y)[8] = xyz[1], (&z)[8] = xyz[2];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        x[c] = px[nodes[c]];
        y[c] = py[nodes[c]];
        z[c] = pz[nodes[c]];
        xv[c] = pxd[nodes[c]];
        yv[c] = pyd[nodes[c]];
        zv[c] = pzd[nodes[c]];
    }
    const double volo = f.volo[el];
    const double v_old = f.v[el];  // read before the stores below may alias it
    // The empty asm takes every node value as an operand, so all the loads are
    // issued before any arithmetic and the element waits for memory once.
    // Without it the compiler issues the velocity loads after the volume
    // arithmetic, and each element waits for two round trips.  The list form
    // (whose node indices are loads themselves) runs faster without it.
    if constexpr (OneTrip) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            asm volatile("" : "+v"(x[c]), "+v"(y[c]), "+v"(z[c]), "+v"(xv[c]), "+v"(yv[c]),
                         "+v"(zv[c]));
        }
        __builtin_amdgcn_s_setprio(1);  // a wave with its data finishes first
    }

#ifdef LULESH_FUSED
    const ElemModes<double> mu = corner_modes(xv), mv = corner_modes(yv), mw = corner_modes(zv);
    const Vec3<double> u[3] = {{mu.a1, mv.a1, mw.a1}, {mu.a2, mv.a2, mw.a2}, {mu.a3, mv.a3, mw.a3}};
    const ElemKinematics r = elem_kinematics(elem_shape(xyz), u, volo, dt);
    f.vnew[el] = r.vnew;
    f.delv[el] = r.vnew - v_old;
    f.arealg[el] = r.arealg;
    f.vdov[el] = r.vdov;
    f.delv_xi[el] = r.delv[0];
    f.delv_eta[el] = r.delv[1];
    f.delv_zeta[el] = r.delv[2];
    f.delx_xi[el] = r.delx[0];
    f.delx_eta[el] = r.delx[1];
    f.delx_zeta[el] = r.delx[2];
    if (r.vnew <= 0.0) {
        raise_error(s, -1);
    }
#else
    // kinematics
    const double volume = elem_volume(x, y, z);
    const double vnew = elem_quot(volume, volo);
    f.vnew[el] = vnew;
    f.delv[el] = vnew - v_old;
    f.arealg[el] = characteristic_length(x, y, z, volume);
    {
        const double dt2 = 0.5 * dt;
        double xh[8], yh[8], zh[8], b[3][4];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            xh[c] = x[c] - dt2 * xv[c];
            yh[c] = y[c] - dt2 * yv[c];
            zh[c] = z[c] - dt2 * zv[c];
        }
        const double det_j = shape_derivatives(xh, yh, zh, b);
        const double inv_det_j = elem_recip(det_j);
        const double dxx = inv_det_j * (b[0][0] * (xv[0] - xv[6]) + b[0][1] * (xv[1] - xv[7]) +
                                        b[0][2] * (xv[2] - xv[4]) + b[0][3] * (xv[3] - xv[5]));
        const double dyy = inv_det_j * (b[1][0] * (yv[0] - yv[6]) + b[1][1] * (yv[1] - yv[7]) +
                                        b[1][2] * (yv[2] - yv[4]) + b[1][3] * (yv[3] - yv[5]));
        const double dzz = inv_det_j * (b[2][0] * (zv[0] - zv[6]) + b[2][1] * (zv[1] - zv[7]) +
                                        b[2][2] * (zv[2] - zv[4]) + b[2][3] * (zv[3] - zv[5]));
        f.vdov[el] = dxx + dyy + dzz;
    }
    if (vnew <= 0.0) {
        raise_error(s, -1);
    }

    // monotonic-Q gradients; each root below is of a sum of squares plus
    // ptiny, so its argument is >= 1e-36 and sqrt_above_tiny is sqrt there
    const double ptiny = 1.e-36;
    const double vol = volo * vnew;
    const double norm = elem_recip(vol + ptiny);
    const double dxj = -0.25 * ((x[0] + x[1] + x[5] + x[4]) - (x[3] + x[2] + x[6] + x[7]));
    const double dyj = -0.25 * ((y[0] + y[1] + y[5] + y[4]) - (y[3] + y[2] + y[6] + y[7]));
    const double dzj = -0.25 * ((z[0] + z[1] + z[5] + z[4]) - (z[3] + z[2] + z[6] + z[7]));
    const double dxi = 0.25 * ((x[1] + x[2] + x[6] + x[5]) - (x[0] + x[3] + x[7] + x[4]));
    const double dyi = 0.25 * ((y[1] + y[2] + y[6] + y[5]) - (y[0] + y[3] + y[7] + y[4]));
    const double dzi = 0.25 * ((z[1] + z[2] + z[6] + z[5]) - (z[0] + z[3] + z[7] + z[4]));
    const double dxk = 0.25 * ((x[4] + x[5] + x[6] + x[7]) - (x[0] + x[1] + x[2] + x[3]));
    const double dyk = 0.25 * ((y[4] + y[5] + y[6] + y[7]) - (y[0] + y[1] + y[2] + y[3]));
    const double dzk = 0.25 * ((z[4] + z[5] + z[6] + z[7]) - (z[0] + z[1] + z[2] + z[3]));
    double ax, ay, az, dxv, dyv, dzv;

    ax = dyi * dzj - dzi * dyj;
    ay = dzi * dxj - dxi * dzj;
    az = dxi * dyj - dyi * dxj;
    f.delx_zeta[el] = elem_quot(vol, sqrt_above_tiny(ax * ax + ay * ay + az * az + ptiny));
    ax *= norm;
    ay *= norm;
    az *= norm;
    dxv = 0.25 * ((xv[4] + xv[5] + xv[6] + xv[7]) - (xv[0] + xv[1] + xv[2] + xv[3]));
    dyv = 0.25 * ((yv[4] + yv[5] + yv[6] + yv[7]) - (yv[0] + yv[1] + yv[2] + yv[3]));
    dzv = 0.25 * ((zv[4] + zv[5] + zv[6] + zv[7]) - (zv[0] + zv[1] + zv[2] + zv[3]));
    f.delv_zeta[el] = ax * dxv + ay * dyv + az * dzv;

    ax = dyj * dzk - dzj * dyk;
    ay = dzj * dxk - dxj * dzk;
    az = dxj * dyk - dyj * dxk;
    f.delx_xi[el] = elem_quot(vol, sqrt_above_tiny(ax * ax + ay * ay + az * az + ptiny));
    ax *= norm;
    ay *= norm;
    az *= norm;
    dxv = 0.25 * ((xv[1] + xv[2] + xv[6] + xv[5]) - (xv[0] + xv[3] + xv[7] + xv[4]));
    dyv = 0.25 * ((yv[1] + yv[2] + yv[6] + yv[5]) - (yv[0] + yv[3] + yv[7] + yv[4]));
    dzv = 0.25 * ((zv[1] + zv[2] + zv[6] + zv[5]) - (zv[0] + zv[3] + zv[7] + zv[4]));
    f.delv_xi[el] = ax * dxv + ay * dyv + az * dzv;

    ax = dyk * dzi - dzk * dyi;
    ay = dzk * dxi - dxk * dzi;
    az = dxk * dyi - dyk * dxi;
    f.delx_eta[el] = elem_quot(vol, sqrt_above_tiny(ax * ax + ay * ay + az * az + ptiny));
    ax *= norm;
    ay *= norm;
    az *= norm;
    dxv = -0.25 * ((xv[0] + xv[1] + xv[5] + xv[4]) - (xv[3] + xv[2] + xv[6] + xv[7]));
    dyv = -0.25 * ((yv[0] + yv[1] + yv[5] + yv[4]) - (yv[3] + yv[2] + yv[6] + yv[7]));
    dzv = -0.25 * ((zv[0] + zv[1] + zv[5] + zv[4]) - (zv[3] + zv[2] + zv[6] + zv[7]));
    f.delv_eta[el] = ax * dxv + ay * dyv + az * dzv;
#endif  // LULESH_FUSED
}

template <class F>
__device__ __forceinline__ void kinematics_q(const F &f, DevScalars *s, int el)
{
    int i, j, k;
    elem_ijk(f, el, i, j, k);
    const int en = f.nx + 1;
    const int n0 = (k * en + j) * en + i;
    const int pl = en * en;
    const int nodes[8] = {n0,      n0 + 1,      n0 + en + 1,      n0 + en,
                          n0 + pl, n0 + pl + 1, n0 + pl + en + 1, n0 + pl + en};
    kinematics_q_nodes<true>(f, s, el, nodes);
}

}  // namespace

__global__ __launch_bounds__(256) void k_kinematics_q(DevFields f, DevScalars *s,
                                                      PhysParams prm)
{
    if (s->active == 0 || s->error != 0) {
        return;
    }
    const int el = int(blockIdx.x) * int(blockDim.x) + int(threadIdx.x);
    if (el < f.num_elem) {
        kinematics_q(f, s, el);
    }
}

// persistent blocks over the element chunks of all members
__global__ __launch_bounds__(256) void k_kinematics_q_batch(const BatchMember *__restrict__ members,
                                                            const BatchWork *__restrict__ work,
                                                            PhysParams prm)
{
    const int n = work->num_chunks;
    const LULESH_AS_GLOBAL int32_t *chunks = (const LULESH_AS_GLOBAL int32_t *)work->chunks;
    for (int c = int(blockIdx.x); c < n; c += int(gridDim.x)) {
        const BatchMember &m = members[chunks[2 * c]];
        if (!member_running(m.s)) {
            continue;
        }
        const int el = chunks[2 * c + 1] + int(threadIdx.x);
        if (el < m.f.num_elem) {
            kinematics_q(global_view(m.f), m.s, el);
        }
    }
}

// The ensemble's element phases with one chunk per block (the default
// launch: a grid of the full chunk list; blocks beyond the current list
// return), without the persistent loop.
__global__ __launch_bounds__(256, 3) void k_kinematics_q_chunks(const BatchMember *__restrict__ members,
                                                             const BatchWork *__restrict__ work,
                                                             PhysParams prm)
{
    const int c = int(blockIdx.x);
    if (c >= work->num_chunks) {
        return;
    }
    const LULESH_AS_GLOBAL int32_t *chunks = (const LULESH_AS_GLOBAL int32_t *)work->chunks;
    const BatchMember &m = members[chunks[2 * c]];
    if (!member_running(m.s)) {
        return;
    }
    const int el = chunks[2 * c + 1] + int(threadIdx.x);
    if (el < m.f.num_elem) {
        kinematics_q(global_view(m.f), m.s, el);
    }
}

namespace {

// limiter of one direction (reference/C/LULESH-OMP.cc:2201-2228)
__device__ __forceinline__ double mono_phi(double self, double delvm,
                                           double delvp, double limiter_mult,
                                           double max_slope)
{
#pragma clang fp contract(off)
    const double ptiny = 1.e-36;
    const double norm = elem_recip(self + ptiny);
    double phi;
    delvm = delvm * norm;
    delvp = delvp * norm;
    phi = .5 * (delvm + delvp);
    delvm *= limiter_mult;
    delvp *= limiter_mult;
    if (delvm < phi) phi = delvm;
    if (delvp < phi) phi = delvp;
    if (phi < 0.) phi = 0.;
    if (phi > max_slope) phi = max_slope;
    return phi;
}

}  // namespace

// ---------------------------------------------------------------------------
// Monotonic Q, EOS, volume update and time constraints of each element.
// k_q_eos_dt_nat (the default) walks the elements in mesh order and shares
// a block's EOS repetitions over its threads; k_q_eos_dt walks them region
// by region (eos_order), so a wavefront mostly shares one repetition count.
// The neighbour across a face is the adjacent element of the structured
// cube; x = 0, y = 0 and z = 0 faces are symmetry planes (neighbour value =
// own value), the far faces free surfaces (neighbour value = 0)
// (reference/C/LULESH-OMP.cc:3153-3171, :2204-2287).  The Courant and hydro
// minima are exact and order independent: each block folds its minimum into
// the cycle's accumulator with an unsigned 64-bit atomic min on the bit
// pattern, and the next kernel boundary applies them (apply_constraints).
// ---------------------------------------------------------------------------
namespace {

// What the monotonic-Q limiter of an element works from
// (reference/C/LULESH-OMP.cc:2182-2320): the limiter values of the three
// directions and, for a compressing element (vdov <= 0), the velocity
// jumps across it (delv * delx, clamped to <= 0) and its density.
struct QInputs {
    double phi[3];
    // the face values the limiter of each direction compares with the
    // element's own (low side, high side), boundary rules applied
    double face[3][2];
    double du[3];
    double rho;
    double vdov, vnew, volo;
    // the element's fields that the EOS and the time constraints read; they
    // are loaded with the limiter's inputs, before the kernel stores anything
    double q_old, v_old, e_old, delv, p_old, arealg;
};

// the rest of the inputs once the limiter values are known
template <class F>
__device__ __forceinline__ void q_inputs_rest(const F &f, int el, double dvxi,
                                              double dveta, double dvzeta, QInputs &in);

template <class F>
__device__ __forceinline__ void q_inputs(const F &f, const PhysParams &prm,
                                         int el, int i, int j, int k, QInputs &in)
{
    const int nx = f.nx;
    const int sy = nx, sz = nx * nx;
    const double dvxi = f.delv_xi[el], dveta = f.delv_eta[el], dvzeta = f.delv_zeta[el];
    // every neighbour is loaded, from the element itself across a boundary
    // face (the value is then replaced), so that no load waits on a branch
    const double xm = f.delv_xi[(i == 0) ? el : el - 1];
    const double xp = f.delv_xi[(i == nx - 1) ? el : el + 1];
    const double ym = f.delv_eta[(j == 0) ? el : el - sy];
    const double yp = f.delv_eta[(j == nx - 1) ? el : el + sy];
    const double zm = f.delv_zeta[(k == 0) ? el : el - sz];
    const double zp = f.delv_zeta[(k == nx - 1) ? el : el + sz];
    q_inputs_rest(f, el, dvxi, dveta, dvzeta, in);
    const double lm = prm.monoq_limiter_mult, ms = prm.monoq_max_slope;
    in.face[0][0] = (i == 0) ? dvxi : xm;
    in.face[0][1] = (i == nx - 1) ? 0.0 : xp;
    in.face[1][0] = (j == 0) ? dveta : ym;
    in.face[1][1] = (j == nx - 1) ? 0.0 : yp;
    in.face[2][0] = (k == 0) ? dvzeta : zm;
    in.face[2][1] = (k == nx - 1) ? 0.0 : zp;
    in.phi[0] = mono_phi(dvxi, in.face[0][0], in.face[0][1], lm, ms);
    in.phi[1] = mono_phi(dveta, in.face[1][0], in.face[1][1], lm, ms);
    in.phi[2] = mono_phi(dvzeta, in.face[2][0], in.face[2][1], lm, ms);
}

// the neighbour value across one face of an unstructured element: own value
// on a symmetry face, 0 on a free face, else the neighbour's
// (reference/C/LULESH-OMP.cc:2201-2287).  The neighbour's value is loaded in
// every case (the mesh builder checks that every neighbour index is an
// element), so that no load waits on the boundary bits.
__device__ __forceinline__ double face_value(double own, double nbr_value, int bc, int symm,
                                             int freeb)
{
    return (bc & symm) ? own : ((bc & freeb) ? 0.0 : nbr_value);
}

__device__ __forceinline__ void q_inputs_u(const DevFields &f, const DevMeshU &m,
                                           const PhysParams &prm, int el, QInputs &in)
{
    const int ne = f.num_elem;
    const int bc = m.elem_bc[el];
    const double dvxi = f.delv_xi[el], dveta = f.delv_eta[el], dvzeta = f.delv_zeta[el];
    const double xm = f.delv_xi[m.nbr[0 * ne + el]], xp = f.delv_xi[m.nbr[1 * ne + el]];
    const double ym = f.delv_eta[m.nbr[2 * ne + el]], yp = f.delv_eta[m.nbr[3 * ne + el]];
    const double zm = f.delv_zeta[m.nbr[4 * ne + el]], zp = f.delv_zeta[m.nbr[5 * ne + el]];
    q_inputs_rest(f, el, dvxi, dveta, dvzeta, in);
    const double lm = prm.monoq_limiter_mult, ms = prm.monoq_max_slope;
    in.phi[0] = mono_phi(dvxi, face_value(dvxi, xm, bc, kBcXiMSymm, kBcXiMFree),
                         face_value(dvxi, xp, bc, kBcXiPSymm, kBcXiPFree), lm, ms);
    in.phi[1] = mono_phi(dveta, face_value(dveta, ym, bc, kBcEtaMSymm, kBcEtaMFree),
                         face_value(dveta, yp, bc, kBcEtaPSymm, kBcEtaPFree), lm, ms);
    in.phi[2] = mono_phi(dvzeta, face_value(dvzeta, zm, bc, kBcZetaMSymm, kBcZetaMFree),
                         face_value(dvzeta, zp, bc, kBcZetaPSymm, kBcZetaPFree), lm, ms);
}

template <class F>
__device__ __forceinline__ void q_inputs_rest(const F &f, int el, double dvxi,
                                              double dveta, double dvzeta, QInputs &in)
{
#pragma clang fp contract(off)
    in.vdov = f.vdov[el];
    in.vnew = f.vnew[el];
    in.volo = f.volo[el];
    in.q_old = f.q[el];
    in.v_old = f.v[el];
    in.e_old = f.e[el];
    in.delv = f.delv[el];
    in.p_old = f.p[el];
    // arealg is read only by a moving element, delx and the mass only by a
    // compressing or resting one (a quiescent element reads neither arealg)
    in.arealg = (in.vdov != 0.) ? f.arealg[el] : 0.0;
    in.du[0] = in.du[1] = in.du[2] = 0.0;
    in.rho = 0.0;
    if (!(in.vdov > 0.)) {
        double dxi = dvxi * f.delx_xi[el];
        double deta = dveta * f.delx_eta[el];
        double dzeta = dvzeta * f.delx_zeta[el];
        if (dxi > 0.) dxi = 0.;
        if (deta > 0.) deta = 0.;
        if (dzeta > 0.) dzeta = 0.;
        in.du[0] = dxi;
        in.du[1] = deta;
        in.du[2] = dzeta;
        in.rho = elem_quot(f.elem_mass[el], in.volo * in.vnew);
    }
}

// The sums of the limiter's linear and quadratic Q over the directions
// (:2289-2316), xi and eta first, and the Q they give.
struct QSums {
    double lin, quad;
};

__device__ __forceinline__ QSums q_sums_xi_eta(double dxi, double phixi, double deta,
                                               double phieta)
{
#pragma clang fp contract(off)
    // rounded alike in both directions
    const double lx = dxi * (1. - phixi), ly = deta * (1. - phieta);
    const double qx = dxi * dxi * madd(-phixi, phixi, 1.);
    const double qy = deta * deta * madd(-phieta, phieta, 1.);
    return {add(lx, ly), add(qx, qy)};
}

__device__ __forceinline__ void q_from_sums(const PhysParams &prm, const QSums &s, double dzeta,
                                            double phizeta, double rho, bool expanding,
                                            double &qlin, double &qquad)
{
#pragma clang fp contract(off)
    if (expanding) {
        qlin = 0.;
        qquad = 0.;
    } else {
        qlin = -prm.qlc_monoq * rho * madd(dzeta, 1. - phizeta, s.lin);
        qquad = prm.qqc_monoq * rho *
                madd(dzeta * dzeta, madd(-phizeta, phizeta, 1.), s.quad);
    }
}

__device__ __forceinline__ void monotonic_q(const PhysParams &prm, const QInputs &in,
                                            double &qlin, double &qquad)
{
    q_from_sums(prm, q_sums_xi_eta(in.du[0], in.phi[0], in.du[1], in.phi[1]), in.du[2],
                in.phi[2], in.rho, in.vdov > 0., qlin, qquad);
}

// What one EOS evaluation of an element reads (the clamped new volume and
// the values of the last cycle), formed once per element.
struct EosIn {
    double vnewc, e_old, delvc, p_old, q_old, qquad, qlin;
};

__device__ __forceinline__ EosConst eos_const(const PhysParams &prm)
{
    EosConst ec;
    ec.e_cut = prm.e_cut;
    ec.p_cut = prm.p_cut;
    ec.q_cut = prm.q_cut;
    ec.eosvmax = prm.eosvmax;
    ec.eosvmin = prm.eosvmin;
    ec.pmin = prm.pmin;
    ec.emin = prm.emin;
    ec.rho0 = prm.refdens;
    ec.unit_rho0 = prm.refdens == 1.0;
    ec.ss_tiny = prm.ss_tiny;
    ec.ss_floor = prm.ss_floor;
    return ec;
}

// The element's side of the EOS before its evaluations: qstop tested on the q of the previous cycle (:2368-2381), the new and old
// relative volumes clamped (:2704-2753; 2.0 clamps vnew in place) and the
// clamped old volume tested.
__device__ __forceinline__ EosIn eos_prepare(DevScalars *s, const PhysParams &prm,
                                             const QInputs &in, double qlin, double qquad)
{
    const double q_old = in.q_old;
    if (q_old > prm.qstop) {
        raise_error(s, -2);
    }
    double vnewc = in.vnew;
    if (prm.eosvmin != 0.) {
        if (vnewc < prm.eosvmin) vnewc = prm.eosvmin;
    }
    if (prm.eosvmax != 0.) {
        if (vnewc > prm.eosvmax) vnewc = prm.eosvmax;
    }
    double vc = in.v_old;
    if (prm.eosvmin != 0.) {
        if (vc < prm.eosvmin) vc = prm.eosvmin;
    }
    if (prm.eosvmax != 0.) {
        if (vc > prm.eosvmax) vc = prm.eosvmax;
    }
    if (vc <= 0.) {
        raise_error(s, -1);
    }
    return EosIn{vnewc, in.e_old, in.delv, in.p_old, q_old, qquad, qlin};
}

// `rep` evaluations of the EOS on the same inputs, as the reference repeats
// them (lulesh-2.0.3/lulesh.cc:2267, :2413-2424).  The inputs pass through an
// empty asm statement at the top of every repetition, so the compiler cannot
// know they are unchanged and computes each repetition in full; they are
// carried from one repetition to the next in the same registers (no copies),
// and every repetition's result is marked as used.
template <bool Unit>
__device__ __forceinline__ EosOut eos_repeat(const EosIn &a, int rep, const EosConst &ec)
{
    double a0 = a.vnewc, a1 = a.e_old, a2 = a.delvc, a3 = a.p_old, a4 = a.q_old;
    double a5 = a.qquad, a6 = a.qlin;
    EosOut o;
    o.p = o.e = o.q = o.ss = 0.0;
    for (int r = 0; r < rep; ++r) {
        asm volatile("" : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5),
                     "+v"(a6));
        o = eos_element<Unit>(a0, a1, a2, a3, a4, a5, a6, ec);
        asm volatile("" ::"v"(o.p), "v"(o.e), "v"(o.q), "v"(o.ss));
    }
    return o;
}

// The element's side after the EOS: p, e, q, ss stored, the volume update
// (UpdateVolumesForElems: 1.0 uses the unclamped vnew, 2.0 the clamped one,
// lulesh-2.0.3/lulesh.cc:2439-2452) and the Courant and hydro candidates
// (:2799-2933).
template <class F>
__device__ __forceinline__ void eos_finish(const F &f, const PhysParams &prm, int el,
                                           const QInputs &in, double vnewc, const EosOut &o,
                                           unsigned long long &cand_c,
                                           unsigned long long &cand_h)
{
    const double vdov = in.vdov, vnew = in.vnew;
    f.p[el] = o.p;
    f.e[el] = o.e;
    f.q[el] = o.q;
    f.ss[el] = o.ss;
    double tmpv = (prm.ic_mode == 1) ? vnew : vnewc;
    if (fabs(tmpv - 1.0) < prm.v_cut) tmpv = 1.0;
    f.v[el] = tmpv;
    if (prm.ic_mode == 2 && vnewc != vnew) {  // memory holds vnew already
        f.vnew[el] = vnewc;
    }
    if (vdov != 0.) {
        const double arealg = in.arealg;
        const double qqc2 = 64.0 * prm.qqc * prm.qqc;
        double dtf = o.ss * o.ss;
        if (vdov < 0.) {
            dtf = madd(qqc2 * arealg * arealg * vdov, vdov, dtf);
        }
        dtf = sqrt(dtf);
        dtf = elem_quot(arealg, dtf);
        cand_c = as_bits(dtf);
        const double dtdvov = elem_quot(prm.dvovmax, fabs(vdov) + 1.e-20);
        cand_h = as_bits(dtdvov);
    }
}

// Everything after ql / qq for one element: qstop, the volume clamps, the
// EOS with the region repetitions, the volume update and the element's
// Courant / hydro candidates.
template <class F>
__device__ __forceinline__ void eos_dt_elem(const F &f, DevScalars *s,
                                            const PhysParams &prm, int el, int rep,
                                            const QInputs &in, double qlin, double qquad,
                                            unsigned long long &cand_c,
                                            unsigned long long &cand_h)
{
    f.ql[el] = qlin;
    f.qq[el] = qquad;
    const EosIn a = eos_prepare(s, prm, in, qlin, qquad);
    const EosConst ec = eos_const(prm);
    EosOut o;
    __builtin_amdgcn_s_setprio(0);  // the repetitions yield to waves still loading
    if (ec.unit_rho0) {
        o = eos_repeat<true>(a, rep, ec);
    } else {
        o = eos_repeat<false>(a, rep, ec);
    }
    __builtin_amdgcn_s_setprio(1);  // stores and the block's reduction
    eos_finish(f, prm, el, in, a.vnewc, o, cand_c, cand_h);
}

// fold the block minima into the cycle's accumulators; they are applied to
// dtcourant / dthydro after the kernel (apply_constraints).  No fence is
// needed: the next kernel on the stream sees the atomics' results.
__device__ __forceinline__ void fold_minima(DevScalars *s, unsigned long long cand_c,
                                            unsigned long long cand_h,
                                            unsigned long long *lds_c,
                                            unsigned long long *lds_h)
{
    const unsigned long long mc = block_min(cand_c, lds_c);
    const unsigned long long mh = block_min(cand_h, lds_h);
    if (threadIdx.x == 0) {
        if (mc < as_bits(kBig)) atomicMin(&s->acc_courant, mc);
        if (mh < as_bits(kBig)) atomicMin(&s->acc_hydro, mh);
    }
}

// one block of 256 elements in schedule order; every thread of the block
// calls it (the minima are reduced over the block)
template <class F>
__device__ __forceinline__ void q_eos_dt_block(const F &f, DevScalars *s,
                                               const PhysParams &prm, int slot,
                                               unsigned long long *lds_c,
                                               unsigned long long *lds_h)
{
    unsigned long long cand_c = as_bits(kBig), cand_h = as_bits(kBig);
    if (slot < f.num_elem) {
        const int el = f.eos_order[slot];
        const int rep = f.eos_rep[slot];
        int i, j, k;
        elem_ijk(f, el, i, j, k);
        QInputs in;
        q_inputs(f, prm, el, i, j, k, in);
        double qlin, qquad;
        monotonic_q(prm, in, qlin, qquad);
        eos_dt_elem(f, s, prm, el, rep, in, qlin, qquad, cand_c, cand_h);
    }
    fold_minima(s, cand_c, cand_h, lds_c, lds_h);
}

}  // namespace

__global__ __launch_bounds__(256) void k_q_eos_dt(DevFields f, DevScalars *s,
                                                  PhysParams prm, int bands)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    // other blocks may raise an error while this one runs: read the flags
    // once per block so that every thread takes the same path to the
    // barriers of the reduction
    if (threadIdx.x == 0) {
        skip = (s->active == 0 || s->error != 0) ? 1 : 0;
    }
    __syncthreads();
    if (skip) {
        return;
    }
    const int chunk = eos_chunk(int(blockIdx.x), int(gridDim.x), bands);
    __builtin_amdgcn_s_setprio(1);  // the element's loads first
    q_eos_dt_block(f, s, prm, chunk * int(blockDim.x) + int(threadIdx.x), lds_c, lds_h);
}

namespace {

// Per block: the EOS inputs of the elements with more than one evaluation,
// by place, and each wave's counts (ExtraDeal).
struct RepLds {
    double in[7][256];
    int cnt[4];
};

// The EOS evaluations of a block's elements beyond each one's first.  The
// thread that owns an element evaluates it once (its result is the
// element's); the others are dealt out over all 256 threads, so a block of
// elements with 1, 2 and 20 repetitions takes ceil(sum(rep - 1) / 256) extra
// passes instead of running every thread 20 times.  An element's evaluations
// all read the same inputs and give the same results: each is computed in
// full (its inputs pass through an empty asm statement) and its result
// marked as used, as the reference repeats the evaluation
// (lulesh-2.0.3/lulesh.cc:2413-2424).  Every thread of the block (256, four
// waves) calls it.
template <bool Unit>
__device__ __forceinline__ void eos_extra_evaluations(const EosIn &a, int extra,
                                                      const int (&classes)[2],
                                                      const EosConst &ec, RepLds &L)
{
    const ExtraDeal deal(extra, classes, L.cnt);
    if (deal.total == 0) {  // the same for every thread of the block
        return;
    }
    if (deal.place >= 0) {
        L.in[0][deal.place] = a.vnewc;
        L.in[1][deal.place] = a.e_old;
        L.in[2][deal.place] = a.delvc;
        L.in[3][deal.place] = a.p_old;
        L.in[4][deal.place] = a.q_old;
        L.in[5][deal.place] = a.qquad;
        L.in[6][deal.place] = a.qlin;
    }
    __syncthreads();
    for (int w = int(threadIdx.x); w < deal.total; w += 256) {
        const int src = deal.owner(w);
        double b0 = L.in[0][src], b1 = L.in[1][src], b2 = L.in[2][src], b3 = L.in[3][src];
        double b4 = L.in[4][src], b5 = L.in[5][src], b6 = L.in[6][src];
        asm volatile("" : "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3), "+v"(b4), "+v"(b5),
                     "+v"(b6));
        const EosOut o = eos_element<Unit>(b0, b1, b2, b3, b4, b5, b6, ec);
        asm volatile("" ::"v"(o.p), "v"(o.e), "v"(o.q), "v"(o.ss));
    }
}

}  // namespace

namespace {

// The EOS of one block of 256 elements in mesh order, el the thread's element
// (valid: it has one), its inputs loaded; every thread of the block calls it
// (the minima are reduced over the block).
template <class F>
__device__ __forceinline__ void eos_nat_block(const F &f, DevScalars *s, const PhysParams &prm,
                                              int el, bool valid, const QInputs &in,
                                              const EosIn &a, int extra,
                                              unsigned long long *lds_c,
                                              unsigned long long *lds_h, RepLds &L)
{
    unsigned long long cand_c = as_bits(kBig), cand_h = as_bits(kBig);
    const EosConst ec = eos_const(prm);
    EosOut o;
    __builtin_amdgcn_s_setprio(0);  // the evaluations yield to waves still loading
    if (ec.unit_rho0) {
        o = eos_repeat<true>(a, 1, ec);
        eos_extra_evaluations<true>(a, extra, f.eos_extra, ec, L);
    } else {
        o = eos_repeat<false>(a, 1, ec);
        eos_extra_evaluations<false>(a, extra, f.eos_extra, ec, L);
    }
    __builtin_amdgcn_s_setprio(1);  // stores and the block's reduction
    if (valid) {
        eos_finish(f, prm, el, in, a.vnewc, o, cand_c, cand_h);
    }
    fold_minima(s, cand_c, cand_h, lds_c, lds_h);
}

// The limiter and the EOS of such a block.
template <class F>
__device__ __forceinline__ void q_eos_dt_nat_block(const F &f, DevScalars *s,
                                                   const PhysParams &prm, int el, bool valid,
                                                   unsigned long long *lds_c,
                                                   unsigned long long *lds_h, RepLds &L)
{
    QInputs in;
    EosIn a{1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int extra = 0;
    if (valid) {
        const int rep = f.rep[el];
        extra = rep - 1;
        int i, j, k;
        elem_ijk(f, el, i, j, k);
        q_inputs(f, prm, el, i, j, k, in);
        double qlin, qquad;
        monotonic_q(prm, in, qlin, qquad);
        f.ql[el] = qlin;
        f.qq[el] = qquad;
        a = eos_prepare(s, prm, in, qlin, qquad);
    }
    eos_nat_block(f, s, prm, el, valid, in, a, extra, lds_c, lds_h, L);
}

}  // namespace

// Monotonic Q, EOS, volume update and time constraints with the elements in
// mesh order, one per thread: each block takes f.eos_elems consecutive
// elements (256, on small domains fewer; eos_block_elems), so the limiter's
// neighbour values and the element's own fields are read in the order they
// lie in memory.  The regions' EOS repetitions are shared
// over each block's threads (eos_extra_evaluations), and the blocks run in
// the order f.eos_blocks gives (costliest first, then the rest in mesh
// order, each XCD on one contiguous part of the mesh; eos_block_order).
__global__ __launch_bounds__(256) void k_q_eos_dt_nat(DevFields f, DevScalars *s,
                                                      PhysParams prm)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    __shared__ RepLds rep_lds;
    if (threadIdx.x == 0) {
        skip = (s->active == 0 || s->error != 0) ? 1 : 0;
    }
    __syncthreads();
    if (skip) {
        return;
    }
    __builtin_amdgcn_s_setprio(1);  // the element's loads first
    const int el = f.eos_blocks[blockIdx.x] * f.eos_elems + int(threadIdx.x);
    q_eos_dt_nat_block(f, s, prm, el, int(threadIdx.x) < f.eos_elems && el < f.num_elem, lds_c,
                       lds_h, rep_lds);
}

#ifdef LULESH_FUSED
namespace {

// Kinematics and the monotonic-Q limiter of the elements, in one sweep.
//
// k_kinematics_q and k_q_eos_dt_nat exchange ten fields of every element
// through memory so that the limiter sees its neighbours' velocity
// gradients: 1298 MB for the two at 150^3, 253 us, the rate a copy reaches.
// Here a block owns TX x TY element columns and nz layers of them and sweeps
// upward, one thread per column.  The gradients of a layer in xi and eta
// reach the neighbouring threads through LDS; the one in zeta waits in its
// own thread for the layer above.  The gradients just outside the tile are
// formed again by 2 (TX + TY) of the threads, those of the layers below and
// above it by every thread.  Out go vnew, the rate of volume change, the
// characteristic length and the two Q terms, which k_eos_dt_nat reads beside
// its own state, and delv; the six gradients only where the cycle is one whose
// fields a caller can read (`store`, or the run ends with it).  Of a cycle
// that turns out to be one because of an error, k_q_gradients forms them again
// from the node copy that s->unstored names.
//
// At 150^3: 475 MB and 135 us here, 358 MB and 83 us for the EOS.  41 M vector
// instructions, half of the time's issue; three waves per SIMD (168 VGPRs)
// wait for each other at the two barriers of a layer.  What did not help:
// the next plane held in registers across a layer (two waves, 142 us, or
// spills, 300 us), tiles of 32 x 8 (145 us) and 64 x 4 (185 us).
template <int TX, int TY>
__device__ __forceinline__ void kinematics_limit_tile(const DevFields &f, DevScalars *s,
                                                      const PhysParams &prm, int nz, bool store,
                                                      int bx, int by, int bz)
{
#pragma clang fp contract(off)
    constexpr int NT = TX * TY, PX = TX + 3, PN = (TX + 3) * (TY + 3);
    constexpr int kHalo = 2 * (TX + TY);
    static_assert(kHalo <= NT, "one halo gradient per thread");
    __shared__ double plane[2][6][PN];      // node planes k and k + 1, one node around the tile
    // the gradients of a layer, one element around the tile: xi in rows of
    // TX + 2, then eta in rows of TX
    constexpr int kEta = TY * (TX + 2);
    __shared__ double grad[kEta + (TY + 2) * TX];
    // what a thread keeps of the layer below until it knows the gradient
    // above: here and not in registers, which decide the occupancy
    __shared__ double below[5][NT];
    const int par = s->cur;
    const double dt = s->deltatime;
    const double *const in[6] = {f.x[par], f.y[par], f.z[par], f.xd[par], f.yd[par], f.zd[par]};
    const int nx = f.nx, en = nx + 1;
    const int tid = int(threadIdx.x), tx = tid % TX, ty = tid / TX;
    const int i0 = bx * TX, j0 = by * TY;
    const int k0 = bz * nz, k1 = min(k0 + nz, nx);  // owned layers [k0, k1)
    const int i = i0 + tx, j = j0 + ty;
    const bool own = i < nx && j < nx;
    store = store || s->last != 0;
    if (tid == 0) {
        s->unstored = store ? 0 : 1 + par;  // every block the same
    }

    constexpr int kSlots = (PN + NT - 1) / NT;
    unsigned gnode[kSlots];  // node of plane 0 in each slot, the nearest outside the domain
#pragma unroll
    for (int r = 0; r < kSlots; ++r) {
        const int idx = min(tid + r * NT, PN - 1);
        const int gi = min(max(i0 - 1 + idx % PX, 0), nx);
        const int gj = min(max(j0 - 1 + idx / PX, 0), nx);
        gnode[r] = unsigned(gj * en + gi);
    }
    double pre[kSlots][6];
    auto fetch_plane = [&](int kp) {
#pragma unroll
        for (int r = 0; r < kSlots; ++r) {
            const unsigned n = unsigned(kp * en * en) + gnode[r];
#pragma unroll
            for (int t = 0; t < 6; ++t) {
                pre[r][t] = load_at(in[t], n);
            }
        }
    };
    auto store_plane = [&](int kp) {
#pragma unroll
        for (int r = 0; r < kSlots; ++r) {
            if ((r + 1) * NT <= PN || tid + r * NT < PN) {
#pragma unroll
                for (int t = 0; t < 6; ++t) {
                    plane[kp & 1][t][tid + r * NT] = pre[r][t];
                }
            }
        }
    };
    // the eight corner values of field t of the element whose first corner
    // is the plane's slot `at`
    auto corners = [&](int k, int t, int at, double (&v)[8]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double *p = plane[(k + h) & 1][t] + at;
            v[4 * h] = p[0];
            v[4 * h + 1] = p[1];
            v[4 * h + 2] = p[PX + 1];
            v[4 * h + 3] = p[PX];
        }
    };
    auto shape = [&](int k, int at) {
        double xyz[3][8];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            corners(k, t, at, xyz[t]);
        }
        return elem_shape(xyz);
    };
    const int at = (ty + 1) * PX + tx + 1;
    const unsigned elem_ji = unsigned(min(j, nx - 1) * nx + min(i, nx - 1));
    auto elem_of = [&](int k) { return unsigned(k * nx * nx) + elem_ji; };

    // The gradients around the tile: number [0, 2 TY) the columns left and
    // right of it (xi), the rest those below and above it (eta).  Every other
    // block gives them to its last threads, so that no SIMD has all of them.
    const int h = (blockIdx.x & 8) ? NT - 1 - tid : tid;
    const bool eta = h >= 2 * TY;
    const int hg = eta ? h - 2 * TY : h;
    const int hside = hg >= (eta ? TX : TY) ? 1 : 0;
    const int hpos = hg - hside * (eta ? TX : TY);
    const int hx = eta ? hpos : (hside ? TX : -1), hy = eta ? (hside ? TY : -1) : hpos;
    const bool halo = h < kHalo && i0 + hx >= 0 && i0 + hx < nx && j0 + hy >= 0 && j0 + hy < nx;
    const int hat = (hy + 1) * PX + hx + 1;
    const unsigned halo_ji = halo ? unsigned((j0 + hy) * nx + i0 + hx) : elem_ji;
    const int hgrad = eta ? kEta + (hy + 1) * TX + hx : hy * (TX + 2) + hx + 1;
    // element fields, loaded one layer ahead
    double volo, v_old, mass, hvolo;
    auto fetch_elem = [&](int k) {
        volo = load_at(f.volo, elem_of(k));
        v_old = load_at(f.v, elem_of(k));
        mass = load_at(f.elem_mass, elem_of(k));
        hvolo = load_at(f.volo, unsigned(k * nx * nx) + halo_ji);
    };

    const double lm = prm.monoq_limiter_mult, ms = prm.monoq_max_slope;
    constexpr double kExpanding = -1.0;  // in place of the density, which q does not need there
    double dz = 0.0;  // the zeta gradient of the layer below the current one
    auto finish = [&](int k, double dz_above) {  // the Q terms of layer k
        const double dz_below = k == 0 ? dz : below[0][tid];
        const double phi = mono_phi(dz, dz_below, dz_above, lm, ms);
        const double rho = below[4][tid];
        double qlin, qquad;
        q_from_sums(prm, QSums{below[1][tid], below[2][tid]}, below[3][tid], phi, rho,
                    rho == kExpanding, qlin, qquad);
        if (own) {
            store_at(f.ql, elem_of(k), qlin);
            store_at(f.qq, elem_of(k), qquad);
        }
    };

    const int kb = max(k0 - 1, 0), ke = min(k1 + 1, nx);  // layers the sweep visits
    fetch_plane(kb);
    store_plane(kb);
    fetch_plane(kb + 1);
    fetch_elem(kb);
    store_plane(kb + 1);
    for (int k = kb; k < ke; ++k) {
        __syncthreads();  // planes k and k + 1 are in LDS
        // the waves with gradients around the tile go first, then those near
        // the barrier (142 -> 133 us at 150^3)
        __builtin_amdgcn_s_setprio(1);
        const bool full = k >= k0 && k < k1;
        if (full && halo) {
            const ElemShape hs = shape(k, hat);
            double u[3];
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                double v[8];
                corners(k, 3 + t, hat, v);
                const ElemModes<double> m = corner_modes(v);
                u[t] = eta ? m.a2 : m.a1;
            }
            grad[hgrad] = elem_gradient(hs.volume, hs.a, Vec3<double>{u[0], u[1], u[2]}, hvolo, eta);
        }
        __builtin_amdgcn_s_setprio(0);
        const ElemShape es = shape(k, at);
        // the positions' registers go to the velocities and the next layer's
        // fields
        __builtin_amdgcn_sched_barrier(0);
        const double volo_k = volo, v_old_k = v_old, mass_k = mass;
        fetch_elem(min(k + 1, ke - 1));
        Vec3<double> u[3];
        {
            double v[8];
            corners(k, 3, at, v);
            const ElemModes<double> mu = corner_modes(v);
            corners(k, 4, at, v);
            const ElemModes<double> mv = corner_modes(v);
            corners(k, 5, at, v);
            const ElemModes<double> mw = corner_modes(v);
            u[0] = {mu.a1, mv.a1, mw.a1};
            u[1] = {mu.a2, mv.a2, mw.a2};
            u[2] = {mu.a3, mv.a3, mw.a3};
        }
        const ElemKinematics r = elem_kinematics(es, u, volo_k, dt);
        const double dz_here = r.delv[2];
        const int gx = ty * (TX + 2) + tx + 1, gy = kEta + (ty + 1) * TX + tx;
        grad[gx] = r.delv[0];
        grad[gy] = r.delv[1];
        __builtin_amdgcn_s_setprio(2);
        __syncthreads();  // gradients staged, plane k read
        if (k > k0) {
            finish(k - 1, dz_here);
        }
        below[0][tid] = dz;
        dz = dz_here;
        if (full) {
            const double xm = grad[gx - 1], xp = grad[gx + 1];
            const double ym = grad[gy - TX], yp = grad[gy + TX];
            const double dx = r.delv[0], dy = r.delv[1];
            const double phix = mono_phi(dx, i == 0 ? dx : xm, i == nx - 1 ? 0.0 : xp, lm, ms);
            const double phiy = mono_phi(dy, j == 0 ? dy : ym, j == nx - 1 ? 0.0 : yp, lm, ms);
            double dux = dx * r.delx[0], duy = dy * r.delx[1];
            double duz = dz * r.delx[2];
            if (dux > 0.) dux = 0.;
            if (duy > 0.) duy = 0.;
            if (duz > 0.) duz = 0.;
            const QSums sums = q_sums_xi_eta(dux, phix, duy, phiy);
            below[1][tid] = sums.lin;
            below[2][tid] = sums.quad;
            below[3][tid] = duz;
            below[4][tid] = r.vdov > 0. ? kExpanding : elem_quot(mass_k, volo_k * r.vnew);
            if (own) {
                const unsigned e = elem_of(k);
                store_at(f.vnew, e, r.vnew);
                store_at(f.vdov, e, r.vdov);
                store_at(f.arealg, e, r.arealg);
                store_at(f.delv, e, r.vnew - v_old_k);
                if (store) {
                    store_at(f.delv_xi, e, r.delv[0]);
                    store_at(f.delv_eta, e, r.delv[1]);
                    store_at(f.delv_zeta, e, r.delv[2]);
                    store_at(f.delx_xi, e, r.delx[0]);
                    store_at(f.delx_eta, e, r.delx[1]);
                    store_at(f.delx_zeta, e, r.delx[2]);
                }
                if (r.vnew <= 0.0) {
                    raise_error(s, -1);
                }
            }
        }
        if (k + 1 < ke) {
            fetch_plane(k + 2);
            store_plane(k + 2);
        }
    }
    if (k1 == nx) {
        finish(nx - 1, 0.0);  // a free surface above
    }
}

// 16 x 16: the tile whose surrounding gradients are exactly one wave's
constexpr int kLimitTX = 16, kLimitTY = 16;

__global__ __launch_bounds__(kLimitTX *kLimitTY, 3) void k_kinematics_limit(DevFields f, DevScalars *s,
                                                                         PhysParams prm, int nz,
                                                                         int store)
{
    __shared__ int skip;
    if (threadIdx.x == 0) {
        skip = (s->active == 0 || s->error != 0) ? 1 : 0;
    }
    __syncthreads();
    if (skip) {
        return;
    }
    const int nbx = (f.nx + kLimitTX - 1) / kLimitTX, nby = (f.nx + kLimitTY - 1) / kLimitTY;
    const int tiles = nbx * nby * ((f.nx + nz - 1) / nz);
    const int t = xcd_order(int(blockIdx.x), tiles);
    if (t >= tiles) {
        return;
    }
    const int r = t / nbx, bz = r / nby;
    kinematics_limit_tile<kLimitTX, kLimitTY>(f, s, prm, nz, store != 0, t - r * nbx,
                                              r - bz * nby, bz);
}

}  // namespace

int kinematics_limit_columns(int nx)
{
    return ((nx + kLimitTX - 1) / kLimitTX) * ((nx + kLimitTY - 1) / kLimitTY);
}

hipError_t launch_kinematics_limit(const DevFields &f, DevScalars *s, const PhysParams &prm,
                                   int nz, bool store, hipStream_t stream)
{
    if (nz < 1) {
        return hipErrorInvalidValue;
    }
    const int64_t tiles = int64_t(kinematics_limit_columns(f.nx)) * ((f.nx + nz - 1) / nz);
    hipLaunchKernelGGL(k_kinematics_limit, dim3(unsigned((tiles + 7) / 8 * 8)),
                       dim3(kLimitTX * kLimitTY), 0, stream, f, s, prm, nz, store ? 1 : 0);
    return hipGetLastError();
}

// The Q gradients that k_kinematics_limit left out, by its functions and so to
// the same bits.
__global__ __launch_bounds__(256) void k_q_gradients(DevFields f, const DevScalars *s)
{
    const int el = int(blockIdx.x) * 256 + int(threadIdx.x);
    if (s->unstored == 0 || el >= f.num_elem) {
        return;
    }
    const int par = s->unstored - 1;
    int i, j, k;
    elem_ijk(f, el, i, j, k);
    const int en = f.nx + 1, n0 = (k * en + j) * en + i;
    const int at[8] = {n0, n0 + 1, n0 + en + 1, n0 + en, n0 + en * en, n0 + en * en + 1,
                       n0 + en * en + en + 1, n0 + en * en + en};
    const double *const in[6] = {f.x[par], f.y[par], f.z[par], f.xd[par], f.yd[par], f.zd[par]};
    double xyz[3][8], vel[3][8];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            xyz[t][c] = in[t][at[c]];
            vel[t][c] = in[3 + t][at[c]];
        }
    }
    const ElemModes<double> mu = corner_modes(vel[0]), mv = corner_modes(vel[1]),
                            mw = corner_modes(vel[2]);
    const Vec3<double> u[3] = {{mu.a1, mv.a1, mw.a1}, {mu.a2, mv.a2, mw.a2}, {mu.a3, mv.a3, mw.a3}};
    // the gradients do not depend on the time step
    const ElemKinematics r = elem_kinematics(elem_shape(xyz), u, f.volo[el], 0.0);
    f.delv_xi[el] = r.delv[0];
    f.delv_eta[el] = r.delv[1];
    f.delv_zeta[el] = r.delv[2];
    f.delx_xi[el] = r.delx[0];
    f.delx_eta[el] = r.delx[1];
    f.delx_zeta[el] = r.delx[2];
}

// EOS, volume update and time constraints after k_kinematics_limit, as
// k_q_eos_dt_nat has them after its limiter.
__global__ __launch_bounds__(256) void k_eos_dt_nat(DevFields f, DevScalars *s, PhysParams prm)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    __shared__ RepLds rep_lds;
    if (threadIdx.x == 0) {
        skip = (s->active == 0 || s->error != 0) ? 1 : 0;
    }
    __syncthreads();
    if (skip) {
        return;
    }
    __builtin_amdgcn_s_setprio(1);  // the element's loads first
    const int el = f.eos_blocks[blockIdx.x] * f.eos_elems + int(threadIdx.x);
    const bool valid = int(threadIdx.x) < f.eos_elems && el < f.num_elem;
    QInputs in;
    EosIn a{1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int extra = 0;
    if (valid) {
        extra = int(f.rep[el]) - 1;
        const unsigned e = unsigned(el);
        const double qlin = load_at(f.ql, e), qquad = load_at(f.qq, e);
        in.vdov = load_at(f.vdov, e);
        in.vnew = load_at(f.vnew, e);
        in.q_old = load_at(f.q, e);
        in.v_old = load_at(f.v, e);
        in.e_old = load_at(f.e, e);
        in.p_old = load_at(f.p, e);
        in.delv = in.vnew - in.v_old;
        in.arealg = (in.vdov != 0.) ? load_at(f.arealg, e) : 0.0;
        a = eos_prepare(s, prm, in, qlin, qquad);
    }
    eos_nat_block(f, s, prm, el, valid, in, a, extra, lds_c, lds_h, rep_lds);
}
#endif  // LULESH_FUSED

// persistent blocks over the element chunks of all members; a chunk lies
// inside one member, so its minima go to that member's accumulators
__global__ __launch_bounds__(256) void k_q_eos_dt_batch(const BatchMember *__restrict__ members,
                                                        const BatchWork *__restrict__ work,
                                                        PhysParams prm)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    __shared__ RepLds rep_lds;
    const int n = work->num_eos;
    const LULESH_AS_GLOBAL int32_t *chunks = (const LULESH_AS_GLOBAL int32_t *)work->eos_chunks;
    for (int c = int(blockIdx.x); c < n; c += int(gridDim.x)) {
        const BatchMember &m = members[chunks[2 * c]];
        __syncthreads();  // the previous chunk's reads of the LDS are done
        if (threadIdx.x == 0) {
            skip = member_running(m.s) ? 0 : 1;
        }
        __syncthreads();
        if (skip) {
            continue;
        }
        __builtin_amdgcn_s_setprio(1);  // the element's loads first
        const int el = chunks[2 * c + 1] + int(threadIdx.x);
        const bool valid = int(threadIdx.x) < work->eos_elems && el < m.f.num_elem;
        q_eos_dt_nat_block(global_view(m.f), m.s, prm, el, valid, lds_c, lds_h, rep_lds);
    }
}

__global__ __launch_bounds__(256) void k_q_eos_dt_chunks(const BatchMember *__restrict__ members,
                                                         const BatchWork *__restrict__ work,
                                                         PhysParams prm)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    __shared__ RepLds rep_lds;
    const int c = int(blockIdx.x);
    if (c >= work->num_eos) {
        return;
    }
    const LULESH_AS_GLOBAL int32_t *chunks = (const LULESH_AS_GLOBAL int32_t *)work->eos_chunks;
    const BatchMember &m = members[chunks[2 * c]];
    if (threadIdx.x == 0) {
        skip = member_running(m.s) ? 0 : 1;
    }
    __syncthreads();
    if (skip) {
        return;
    }
    __builtin_amdgcn_s_setprio(1);  // the element's loads first
    const int el = chunks[2 * c + 1] + int(threadIdx.x);
    const bool valid = int(threadIdx.x) < work->eos_elems && el < m.f.num_elem;
    q_eos_dt_nat_block(global_view(m.f), m.s, prm, el, valid, lds_c, lds_h, rep_lds);
}

// ---------------------------------------------------------------------------
// The learned closure, in one of two forms (LearnedForm).
//
// Factors (form 0): the network sees twelve dimensionless inputs formed
// from what the monotonic limiter works from and its result:
//   0-2   the limiter values phi of the xi, eta, zeta directions
//   3-5   the velocity jumps du (delv * delx, <= 0) over the sound speed c,
//         as du / (c + |du|)
//   6-8   delx of each direction over their mean hbar
//   9     vdov * hbar / (c + |vdov| hbar)
//   10    log of the relative volume vnew (the density is m / (V0 vnew))
//   11    log of the sound speed c of the last EOS evaluation
// and returns two factors on the monotonic limiter's linear and quadratic
// Q of the element, ql = m_l ql_limiter, qq = m_q qq_limiter.
//
// Stand-in (form 1): the network takes the limiter's place.  It sees the
// limiter's inputs rather than its result:
//   0-5   the velocity gradients across the element's faces relative to its
//         own, r = delv_face / delv (low and high face of xi, eta, zeta; the
//         boundary rules of the limiter applied), as r / (1 + |r|)
//   6-8   the velocity jumps du / (c + |du|)
//   9     vdov * hbar / (c + |vdov| hbar)
//   10    log of the relative volume vnew (the density is m / (V0 vnew))
//   11    log of the sound speed c
// and its two outputs are the linear and quadratic limiting factors
// themselves: ql = -qlc rho m_l sum du, qq = qqc rho m_q sum du^2 (the
// plain limiter's factors are sum du (1 - phi) / sum du and
// sum du^2 (1 - phi^2) / sum du^2); the limiter is evaluated only for the
// elements that fall back to it.
//
// In both forms each output is clamped to [0, 3], and an element keeps the
// plain limiter when an input lies more than z_max standard deviations from
// the training mean, when its volume or energy is not positive, or when it
// has no compression to limit.
// ---------------------------------------------------------------------------
namespace {

__device__ __forceinline__ void learned_inputs(const DevFields &f, const QInputs &in,
                                               int el, int form, float feat[kMlpIn],
                                               double &ql_unlim, double &qq_unlim,
                                               bool &usable)
{
    const double c = f.ss[el];
    const double hbar = (f.delx_xi[el] + f.delx_eta[el] + f.delx_zeta[el]) * (1.0 / 3.0);
    const double delx[3] = {f.delx_xi[el], f.delx_eta[el], f.delx_zeta[el]};
    const double self[3] = {f.delv_xi[el], f.delv_eta[el], f.delv_zeta[el]};
    if (form == 0) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            feat[d] = float(in.phi[d]);
            feat[3 + d] = float(in.du[d] / (c + fabs(in.du[d]) + 1e-300));
            feat[6 + d] = float(delx[d] / hbar);
        }
    } else {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double norm = 1.0 / (self[d] + 1.e-36);
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const double r = in.face[d][side] * norm;
                feat[2 * d + side] = float(r / (1.0 + fabs(r)));
            }
            feat[6 + d] = float(in.du[d] / (c + fabs(in.du[d]) + 1e-300));
        }
    }
    feat[9] = float(in.vdov * hbar / (c + fabs(in.vdov) * hbar + 1e-300));
    feat[10] = float(log(in.vnew > 0.0 ? in.vnew : 1.0));
    feat[11] = float(log(c > 0.0 ? c : 1e-300));
    const double sdu = in.du[0] + in.du[1] + in.du[2];
    const double sdu2 = in.du[0] * in.du[0] + in.du[1] * in.du[1] + in.du[2] * in.du[2];
    ql_unlim = -in.rho * sdu;
    qq_unlim = in.rho * sdu2;
    usable = !(in.vdov > 0.) && sdu < 0.0 && in.vnew > 0.0 && f.e[el] >= 0.0 &&
             hbar > 0.0 && c > 0.0;
}

}  // namespace

// features of every element for training: feat[el][12] and
// q[el][4] = (unlimited ql / qlc, unlimited qq / qqc, plain ql, plain qq);
// the unlimited values are 0 where the element has no compression
__global__ __launch_bounds__(256) void k_q_features(DevFields f, PhysParams prm, int form,
                                                    float *feat, double *q)
{
    const int el = int(blockIdx.x) * int(blockDim.x) + int(threadIdx.x);
    if (el >= f.num_elem) {
        return;
    }
    int i, j, k;
    elem_ijk(f, el, i, j, k);
    QInputs in;
    q_inputs(f, prm, el, i, j, k, in);
    double qlin, qquad;
    monotonic_q(prm, in, qlin, qquad);
    float x[kMlpIn];
    double ql_u, qq_u;
    bool usable;
    learned_inputs(f, in, el, form, x, ql_u, qq_u, usable);
    for (int t = 0; t < kMlpIn; ++t) {
        feat[size_t(el) * kMlpIn + t] = x[t];
    }
    q[size_t(el) * 4 + 0] = usable ? ql_u : 0.0;
    q[size_t(el) * 4 + 1] = usable ? qq_u : 0.0;
    q[size_t(el) * 4 + 2] = qlin;
    q[size_t(el) * 4 + 3] = qquad;
}

namespace {

// The Q terms of one wave's 64 elements with the learned closure in place of
// the limiter, the network evaluated on the matrix cores; every lane of the
// wave calls it (valid: the lane has an element).
__device__ __forceinline__ void learned_q_wave(const DevFields &f, const PhysParams &prm,
                                               const MlpFrags &F, float z_max, int form,
                                               MlpWaveLds &L, int el, bool valid, QInputs &in,
                                               double &qlin, double &qquad)
{
    const int lane = int(threadIdx.x) & 63;
    double ql_u = 0.0, qq_u = 0.0;
    qlin = 0.0;
    qquad = 0.0;
    bool use_net = false;
    float x[kMlpIn];
#pragma unroll
    for (int t = 0; t < kMlpIn; ++t) {
        x[t] = 0.f;
    }
    if (valid) {
        int i, j, k;
        elem_ijk(f, el, i, j, k);
        q_inputs(f, prm, el, i, j, k, in);
        if (form == 0) {
            monotonic_q(prm, in, qlin, qquad);
        }
        learned_inputs(f, in, el, form, x, ql_u, qq_u, use_net);
    }
    // standardise; out-of-range inputs keep the plain limiter
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        float z = 0.f;
        if (t < kMlpIn) {
            z = (x[t] - F.in_mean[t]) * F.in_inv_std[t];
            if (!(fabsf(z) <= z_max)) {
                use_net = false;
                z = 0.f;
            }
        }
        L.x[lane][t] = to_bf16(z);
    }
    __builtin_amdgcn_wave_barrier();
    mlp_forward_wave(F, L, lane);
    if (use_net) {
        const float ml = fminf(fmaxf(L.y[lane][0], 0.f), 3.f);
        const float mq = fminf(fmaxf(L.y[lane][1], 0.f), 3.f);
        if (form == 0) {
            qlin = double(ml) * qlin;
            qquad = double(mq) * qquad;
        } else {
            // the network's limiting factors on the unlimited sums
            qlin = prm.qlc_monoq * (double(ml) * ql_u);
            qquad = prm.qqc_monoq * (double(mq) * qq_u);
        }
    } else if (valid && form != 0) {
        monotonic_q(prm, in, qlin, qquad);  // the fallback: the plain limiter
    }
}

}  // namespace

// k_q_eos_dt with the learned closure, one wave per block (20 KB of LDS): four
// to a block left a CU four waves, one to a block seven.  150^3 step 820 -> 788
// us, 100^3 264 -> 246.
__global__ __launch_bounds__(64) void k_q_eos_dt_learned(DevFields f, DevScalars *s,
                                                         PhysParams prm, const MlpFrags *net,
                                                         float z_max, int form)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ MlpWaveLds L;
    // one wave: its lanes see the same flags
    if (s->active == 0 || s->error != 0) {
        return;
    }
    const int slot = (int(gridDim.x) - 1 - int(blockIdx.x)) * 64 + int(threadIdx.x);
    const bool valid = slot < f.num_elem;
    int el = 0, rep = 0;
    if (valid) {
        el = f.eos_order[slot];
        rep = f.eos_rep[slot];
    }
    QInputs in;
    double qlin, qquad;
    learned_q_wave(f, prm, *net, z_max, form, L, el, valid, in, qlin, qquad);
    unsigned long long cand_c = as_bits(kBig), cand_h = as_bits(kBig);
    if (valid) {
        eos_dt_elem(f, s, prm, el, rep, in, qlin, qquad, cand_c, cand_h);
    }
    fold_minima(s, cand_c, cand_h, lds_c, lds_h);
}

// The same for small domains, in mesh order, 64 elements per block, their
// repetitions shared by its four waves as in k_q_eos_dt_nat: on a chip that
// is not full the launch lasts as long as the 20 evaluations of one wave.
// Steps in us with k_q_eos_dt_learned and with this: 10^3 31.4, 24.0; 33^3 37.9,
// 32.0; 36^3 46.8, 41.1; 38^3 48.2, 48.5; 45^3 59.6, 63.4.
__global__ __launch_bounds__(256) void k_q_eos_dt_learned_nat(DevFields f, DevScalars *s,
                                                              PhysParams prm,
                                                              const MlpFrags *net, float z_max,
                                                              int form)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    __shared__ MlpWaveLds L;
    __shared__ RepLds rep_lds;
    if (threadIdx.x == 0) {
        skip = (s->active == 0 || s->error != 0) ? 1 : 0;
    }
    __syncthreads();
    if (skip) {
        return;
    }
    const int el = int(blockIdx.x) * 64 + int(threadIdx.x);
    const bool valid = int(threadIdx.x) < 64 && el < f.num_elem;
    QInputs in;
    EosIn a{1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int extra = 0;
    if (wave_uniform(int(threadIdx.x) >> 6) == 0) {
        double qlin, qquad;
        learned_q_wave(f, prm, *net, z_max, form, L, el, valid, in, qlin, qquad);
        if (valid) {
            extra = int(f.rep[el]) - 1;
            f.ql[el] = qlin;
            f.qq[el] = qquad;
            a = eos_prepare(s, prm, in, qlin, qquad);
        }
    }
    eos_nat_block(f, s, prm, el, valid, in, a, extra, lds_c, lds_h, rep_lds);
}

// ---------------------------------------------------------------------------
// Unstructured meshes: the same element phases, nodes and face neighbours
// from the mesh's lists
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_kinematics_q_u(DevFields f, DevMeshU m,
                                                        DevScalars *s, PhysParams prm)
{
    if (s->active == 0 || s->error != 0) {
        return;
    }
    const int el = mesh_block(f.num_elem, int(gridDim.x)) * int(blockDim.x) + int(threadIdx.x);
    const int ne = f.num_elem;
    if (el < ne) {
        int nodes[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            nodes[c] = m.nodelist[c * ne + el];
        }
        kinematics_q_nodes<false>(f, s, el, nodes);
    }
}

__global__ __launch_bounds__(256) void k_q_eos_dt_u(DevFields f, DevMeshU m, DevScalars *s,
                                                    PhysParams prm)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    if (threadIdx.x == 0) {
        skip = (s->active == 0 || s->error != 0) ? 1 : 0;
    }
    __syncthreads();
    if (skip) {
        return;
    }
    const int slot = mesh_block(f.num_elem, int(gridDim.x)) * int(blockDim.x) + int(threadIdx.x);
    unsigned long long cand_c = as_bits(kBig), cand_h = as_bits(kBig);
    if (slot < f.num_elem) {
        const int el = f.eos_order[slot];
        const int rep = f.eos_rep[slot];
        QInputs in;
        q_inputs_u(f, m, prm, el, in);
        double qlin, qquad;
        monotonic_q(prm, in, qlin, qquad);
        eos_dt_elem(f, s, prm, el, rep, in, qlin, qquad, cand_c, cand_h);
    }
    fold_minima(s, cand_c, cand_h, lds_c, lds_h);
}

// applies the minima of the last cycle: 2.0 starts every cycle from 1e20
// (lulesh-2.0.3/lulesh.cc:2616-2620); 1.0 keeps the previous constraint when
// no element gave one (reference/C/LULESH-OMP.cc:2867-2871)
__global__ void k_dt_finish(const DevScalars *from, DevScalars *s, int ic_mode)
{
    if (threadIdx.x == 0) {
        DevScalars t = *from;
        apply_constraints(&t, ic_mode);
        *s = t;
    }
}

// the same for every member, and the count of members that have cycles
// left (not failed, time < stoptime, cycle < max_cycles); one block
__global__ void k_dt_finish_batch(const BatchMember *members, BatchWork *work,
                                  int ic_mode)
{
    __shared__ int pending;
    if (threadIdx.x == 0) {
        pending = 0;
    }
    __syncthreads();
    const int n = work->num_members;
    int mine = 0;
    for (int m = int(threadIdx.x); m < n; m += int(blockDim.x)) {
        DevScalars *s = members[m].s;
        apply_constraints(s, ic_mode);
        if (s->error == 0 && s->time < s->stoptime && s->cycle < s->max_cycles) {
            ++mine;
        }
    }
    if (mine) {
        atomicAdd(&pending, mine);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        work->num_pending = pending;
    }
}

// device math probe: op 0 = lulesh_cbrt(a), 1 = sqrt(a), 2 = the element
// arithmetic's quotient a / b (elem_quot: a divide here, the refined
// reciprocal in the fused build), 3 = sqrt_above_tiny(a) (the EOS's square
// root), 4 = the hourglass coefficient's a / cbrt(b) (elem_over_cbrt)
__global__ void k_device_math(int op, int n, const double *a, const double *b,
                              double *out)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) {
        return;
    }
    if (op == 0) {
        out[t] = lulesh_cbrt(a[t]);
    } else if (op == 1) {
        out[t] = sqrt(a[t]);
    } else if (op == 3) {
        out[t] = sqrt_above_tiny(a[t]);
    } else if (op == 4) {
        out[t] = elem_over_cbrt(a[t], b[t]);
    } else {
        out[t] = elem_quot(a[t], b[t]);
    }
}

LULESH_VARIANT_END
}  // namespace lulesh
