// lulesh_mixed.hip -- the mixed-precision form of the cycle.
//
// Same phases, launch structure and data flow as the float64 step
// (lulesh_force.hip, lulesh_kernels.hip), with the element-local arithmetic
// of the stress integration, the hourglass control, the monotonic Q and the
// equation of state in float32.  What stays float64:
//   - node coordinates, velocities, masses and the whole nodal update;
//   - element volumes: the Jacobian determinant of the VolumeError check,
//     the element volume behind vnew, and the half-step Jacobian of the
//     velocity gradient (cancellation in these differences of coordinates
//     is where float32 would lose the most);
//   - the energy update of the EOS (e and its three increments);
//   - the Courant / hydro reductions (each element's candidate is widened
//     to float64 before the minimum).
// Float32 geometry is formed on coordinates relative to the element's node
// 0 (differences taken in float64, then rounded): every quantity it feeds
// is translation invariant, and the local coordinates keep the relative
// precision of the element size rather than of the domain size.
// Multiply-adds may be fused here; reciprocals, square roots and the cube
// root use the hardware float32 approximations (1 ulp).
#define LULESH_MIXED_TU 1
#include "lulesh_kernels.hpp"

#include "lulesh_elem.hpp"
#include "lulesh_modal.hpp"

#pragma clang fp contract(fast)

namespace lulesh {

namespace {

constexpr double kBig = 1.0e+20;

__device__ __forceinline__ float frcp(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ __forceinline__ float frsq(float v) { return __builtin_amdgcn_rsqf(v); }
__device__ __forceinline__ float fsqrt(float v) { return __builtin_amdgcn_sqrtf(v); }
// cube root of a positive normal float: 2^(log2(v) / 3)
__device__ __forceinline__ float fcbrt(float v)
{
    return __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(v) * (1.0f / 3.0f));
}

__device__ __forceinline__ unsigned long long as_bits(double v)
{
    return static_cast<unsigned long long>(__double_as_longlong(v));
}

__device__ __forceinline__ void raise_error(DevScalars *s, int code)
{
    atomicCAS(&s->error, 0, code);
}

__device__ __forceinline__ void elem_ijk(const DevFieldsMixed &f, int el, int &i, int &j,
                                         int &k)
{
    const unsigned q1 = fast_div(unsigned(el), f.div_nx);
    i = el - int(q1) * f.nx;
    const unsigned q2 = fast_div(q1, f.div_nx);
    j = int(q1) - int(q2) * f.nx;
    k = int(q2);
}

// ---------------------------------------------------------------------------
// Force sweep: the tiling of sweep_tile (lulesh_force.hip), with an element's
// stress and hourglass forces formed in its modes (lulesh_modal.hpp) in
// float32, each kind by itself.  They meet in float64: added there, turned
// into corner forces, staged and summed over a node's eight corners, the
// layers' two faces as modes within the thread, as in the fused float64 sweep.
//
// Against the two kinds corner by corner, staged one after the other and
// summed in float32: 120^3 step 193 -> 174 us, 150^3 373 -> 341, 91^3 97 -> 85
// (per thread and layer 892 instead of 1629 vector instructions, two barriers
// instead of six).  With the kinds added in float32 the times are the same
// (120^3 173.5, 150^3 341.1, 91^3 84.6; 200^3 810 against 828), but the small kind lost what an ulp of
// the large one holds.  Errors against the float64 run, relative to the form
// corner by corner, in the geometric mean over 76 runs of 30^3 to 130^3 to
// t = 1e-2: origin energy 1.04 (added in float32 1.11), total energy 1.07
// (1.06), x 0.93, xd 1.02, e 1.00 (1.10), p 1.00, q 0.92, v 1.02 (1.15), ss
// 1.01; over 36 stretches of 84 to 920 cycles on 20^3 to 200^3: time 0.73
// (0.93), origin energy 0.99 (1.22), x 0.74 (1.08), xd 0.80 (1.13), e 0.92
// (1.13), p 0.77 (1.08), v 0.84 (1.06).  Single runs scatter by half.  120^3:
// origin energy 2.4e-6 (6.6e-6; corner by corner 2.5e-6).
// ---------------------------------------------------------------------------
template <int TX, int TY>
__device__ __forceinline__ void sweep_tile_mixed(const DevFieldsMixed &f,
                                                 const DevScalars *from, DevScalars *s,
                                                 const PhysParams &prm, int nz, int bx,
                                                 int by, int bz)
{
    constexpr int NT = TX * TY;
    constexpr int PX = TX + 1;
    constexpr int PN = (TX + 1) * (TY + 1);
    __shared__ double plane[2][6][PN];
    __shared__ double side[3][3][NT];  // forces on corners 1, 2, 3 of each thread's face
    __shared__ int s_go, s_par;
    __shared__ double s_dt;

    const int tid = threadIdx.x;
    if (tid == 0) {
        const CycleStart c =
            start_cycle(from, s, prm.ic_mode, bx == 0 && by == 0 && bz == 0);
        s_go = c.go;
        s_par = c.par;
        s_dt = c.dt;
    }
    __syncthreads();
    if (!s_go) {
        return;
    }
    const int par = s_par;
    const double dt = s_dt;
    const int nx = f.nx;
    const int en = nx + 1;
    const double *__restrict__ in[6] = {f.x[par ^ 1], f.y[par ^ 1], f.z[par ^ 1],
                                        f.xd[par ^ 1], f.yd[par ^ 1], f.zd[par ^ 1]};
    const int tx = tid % TX;
    const int ty = tid / TX;
    const int i0 = bx * (TX - 1);
    const int j0 = by * (TY - 1);
    const int kc0 = bz * nz;
    const int kc1 = min(kc0 + nz, en);
    const int ie = i0 - 1 + tx;
    const int je = j0 - 1 + ty;
    const bool col_valid = ie >= 0 && ie < nx && je >= 0 && je < nx;
    const bool owner = tx >= 1 && ty >= 1 && ie <= nx && je <= nx;
    const float hg = prm.hgcoef > 0.0 ? float(-prm.hgcoef * 0.01) : 0.0f;

    constexpr int kSlots = (PN + NT - 1) / NT;
    int gnode[kSlots];
#pragma unroll
    for (int r = 0; r < kSlots; ++r) {
        const int idx = tid + r * NT;
        const int lx = idx % PX;
        const int ly = idx / PX;
        const int gi = i0 - 1 + lx;
        const int gj = j0 - 1 + ly;
        gnode[r] = (idx < PN && gi >= 0 && gi <= nx && gj >= 0 && gj <= nx)
                       ? gj * en + gi
                       : -1;
    }
    const int plane_stride = en * en;
    double pre[kSlots][6];
    auto fetch_plane = [&](int kp) {
#pragma unroll
        for (int r = 0; r < kSlots; ++r) {
            if (gnode[r] >= 0) {
                const int n = kp * plane_stride + gnode[r];
#pragma unroll
                for (int fld = 0; fld < 6; ++fld) {
                    pre[r][fld] = in[fld][n];
                }
            } else {
#pragma unroll
                for (int fld = 0; fld < 6; ++fld) {
                    pre[r][fld] = 0.0;
                }
            }
        }
    };
    auto store_plane = [&](int slot) {
#pragma unroll
        for (int r = 0; r < kSlots; ++r) {
            const int idx = tid + r * NT;
            if (idx < PN) {
#pragma unroll
                for (int fld = 0; fld < 6; ++fld) {
                    plane[slot][fld][idx] = pre[r][fld];
                }
            }
        }
    };
    const int base = ty * PX + tx;
    const int nodeoff[4] = {base, base + 1, base + PX + 1, base + PX};

    double top[3][4] = {};  // forces on the face of plane k from the layer below, as modes
    // element fields of the next layer and the owned node's mass of the next
    // plane, loaded one iteration ahead (see sweep_tile)
    float pq_pre[3] = {0.f, 0.f, 0.f};        // p, q, ss
    double vm_pre[3] = {0.0, 0.0, 0.0};       // v, volo, elemMass
    double mass_pre = 1.0;
    auto fetch_elem = [&](int kk) {
        if (kk < nx && col_valid) {
            const int e = (kk * nx + je) * nx + ie;
            pq_pre[0] = f.p[e];
            pq_pre[1] = f.q[e];
            pq_pre[2] = f.ss[e];
            vm_pre[0] = f.v[e];
            vm_pre[1] = f.volo[e];
            vm_pre[2] = f.elem_mass[e];
        }
    };
    auto fetch_mass = [&](int kk) {
        if (owner && kk >= kc0 && kk < kc1) {
            mass_pre = f.nodal_mass[(kk * en + je) * en + ie];
        }
    };
    // float64 corner values of component t between planes lo and hi
    auto corner8 = [&](int lo, int t, double *X) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            X[c] = plane[lo][t][nodeoff[c]];
            X[c + 4] = plane[lo ^ 1][t][nodeoff[c]];
        }
    };
    // their modes in float32: no mode changes with a uniform value, so they are
    // taken relative to corner 0
    auto modes8 = [](const double *X) {
        float x[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            x[c] = float(X[c] - X[0]);
        }
        return elem_modes(face_modes(x[0], x[1], x[2], x[3]),
                          face_modes(x[4], x[5], x[6], x[7]));
    };
    const int kbeg = (kc0 > 0) ? kc0 - 1 : 0;
    fetch_elem(kbeg);
    fetch_mass(kbeg);
    fetch_plane(kbeg);
    store_plane(kbeg & 1);
    fetch_plane(kbeg + 1);  // kbeg < nx
    store_plane((kbeg + 1) & 1);
    if (kbeg + 1 < nx && kbeg + 1 < kc1) {
        fetch_plane(kbeg + 2);
    }
    __syncthreads();
    // Iteration k: the element layer between planes k and k + 1 (both in LDS,
    // plane k + 2 on its way), then the nodes of plane k.  Wave priority rises
    // towards a barrier, as in the float64 sweep.
    for (int k = kbeg; k < kc1; ++k) {
        const bool layer = k < nx;
        __builtin_amdgcn_s_setprio(1);
        const int lo = k & 1;
        const bool finalize = owner && k >= kc0;
        const bool compute = layer && col_valid;
        const float ep = pq_pre[0], eq = pq_pre[1], ess = pq_pre[2];
        const double ev = vm_pre[0], evolo = vm_pre[1], emass = vm_pre[2];
        const double nmass = mass_pre;
        fetch_elem(k + 1);
        fetch_mass(k + 1);

        // ---- stress and hourglass forces, in the element's modes ----
        double face[3][4];  // on the face of plane k, both layers
#pragma unroll
        for (int t = 0; t < 3; ++t) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                face[t][c] = top[t][c];
                top[t][c] = 0.0;
            }
        }
        if (compute) {
            ElemModes<float> xm, ym, zm;
            {
                double X[8], Y[8], Z[8];
                corner8(lo, 0, X);
                corner8(lo, 1, Y);
                corner8(lo, 2, Z);
                // VolumeError on the Jacobian volume, then on v, which the
                // reference tests for every element before it looks at
                // hgcoef (reference/C/LULESH-OMP.cc:1579-1584, :1540-1543)
                if (jacobian_volume(X, Y, Z) <= 0.0 || ev <= 0.0) {
                    raise_error(s, -1);
                }
                xm = modes8(X);
                ym = modes8(Y);
                zm = modes8(Z);
            }
            const float determ = float(evolo * ev);
            ForceShape<float> sh;
            force_shape(xm, ym, zm, frcp(determ), sh);
            const float coef = hg * ess * float(emass) * frcp(fcbrt(determ));
            const double press64 = (double(ep) + double(eq)) * 0.015625;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                double U[8];
                corner8(lo, 3 + t, U);
                // the hourglass forces; the stress joins them in float64
                const ElemModes<float> h =
                    force_modes(sh, 0.0f, 0.0f, 0.0f, 0.0f, coef, modes8(U));
                const double n1 = t == 0 ? sh.n[0].x : t == 1 ? sh.n[0].y : sh.n[0].z;
                const double n2 = t == 0 ? sh.n[1].x : t == 1 ? sh.n[1].y : sh.n[1].z;
                const double n3 = t == 0 ? sh.n[2].x : t == 1 ? sh.n[2].y : sh.n[2].z;
                const double a1 = fused_madd(press64, n1, double(h.a1));
                const double a2 = fused_madd(press64, n2, double(h.a2));
                const double a3 = fused_madd(press64, n3, double(h.a3));
                const double h1 = h.h1, h2 = h.h2, h3 = h.h3, h4 = h.h4;
                face[t][0] -= a3;
                face[t][1] += a1 - h2;
                face[t][2] += a2 - h1;
                face[t][3] += h3 - h4;
                top[t][0] = a3;
                top[t][1] = a1 + h2;
                top[t][2] = a2 + h1;
                top[t][3] = h3 + h4;
            }
        }
        __builtin_amdgcn_s_setprio(2);
        // corner 0 stays, corners 1, 2, 3 go to the threads whose node they are
        double F[3], own[6];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const double ap = face[t][0] + face[t][1], am = face[t][0] - face[t][1];
            const double bp = face[t][2] + face[t][3], bm = face[t][2] - face[t][3];
            F[t] = am - bm;
            side[t][0][tid] = ap - bp;
            side[t][1][tid] = ap + bp;
            side[t][2][tid] = am + bm;
            own[t] = plane[lo][t][base];
            own[3 + t] = plane[lo][3 + t][base];
        }
        __syncthreads();  // the faces are staged, plane k is read
        // ---- acceleration, symmetry planes, velocity, position: float64 ----
        if (finalize) {
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                F[t] += (side[t][1][tid - TX - 1] + side[t][2][tid - TX]) + side[t][0][tid - 1];
            }
            const int n = (k * en + je) * en + ie;
            const double minv = 1.0 / nmass;
            double xdd = F[0] * minv;
            double ydd = F[1] * minv;
            double zdd = F[2] * minv;
            if (ie == 0) xdd = 0.0;
            if (je == 0) ydd = 0.0;
            if (k == 0) zdd = 0.0;
            double xd = own[3] + xdd * dt;
            if (fabs(xd) < prm.u_cut) xd = 0.0;
            double yd = own[4] + ydd * dt;
            if (fabs(yd) < prm.u_cut) yd = 0.0;
            double zd = own[5] + zdd * dt;
            if (fabs(zd) < prm.u_cut) zd = 0.0;
            f.xd[par][n] = xd;
            f.yd[par][n] = yd;
            f.zd[par][n] = zd;
            f.x[par][n] = own[0] + xd * dt;
            f.y[par][n] = own[1] + yd * dt;
            f.z[par][n] = own[2] + zd * dt;
        }
        if (k + 1 < nx && k + 1 < kc1) {
            store_plane(lo);  // plane k + 2
            if (k + 2 < nx && k + 2 < kc1) {
                fetch_plane(k + 3);
            }
        }
        __syncthreads();  // plane k + 2 is in LDS, the faces are read
    }
}

// tiles in the order of k_force_sweep, whose reason holds here too
template <int TX, int TY, int W>
__global__ __launch_bounds__(TX *TY, W) void k_force_sweep_mixed(DevFieldsMixed f,
                                                              const DevScalars *__restrict__ from,
                                                              DevScalars *s,
                                                              PhysParams prm, int nz)
{
    const int nbx = (f.nx + TX - 1) / (TX - 1), nby = (f.nx + TY - 1) / (TY - 1);
    const int tiles = nbx * nby * ((f.nx + nz) / nz);
    const int t = xcd_order(int(blockIdx.x), tiles);
    if (t >= tiles) {
        return;
    }
    const int r = t / nbx, bz = r / nby;
    sweep_tile_mixed<TX, TY>(f, from, s, prm, nz, t - r * nbx, r - bz * nby, bz);
}

template <int TX, int TY, int W>
hipError_t launch_mixed_shape(int nz, const DevFieldsMixed &f, const DevScalars *from,
                              DevScalars *s, const PhysParams &prm, hipStream_t stream)
{
    const int64_t tiles = int64_t((f.nx + TX - 1) / (TX - 1)) *
                          ((f.nx + TY - 1) / (TY - 1)) * ((f.nx + nz) / nz);
    hipLaunchKernelGGL((k_force_sweep_mixed<TX, TY, W>), dim3(unsigned((tiles + 7) / 8 * 8)),
                       dim3(TX * TY), 0, stream, f, from, s, prm, nz);
    return hipGetLastError();
}

// limiter of one direction (reference/C/LULESH-OMP.cc:2201-2228), float32
__device__ __forceinline__ float mono_phi(float self, float delvm, float delvp,
                                          float limiter_mult, float max_slope)
{
    const float norm = frcp(self + 1.e-36f);
    delvm = delvm * norm;
    delvp = delvp * norm;
    float phi = .5f * (delvm + delvp);
    delvm *= limiter_mult;
    delvp *= limiter_mult;
    if (delvm < phi) phi = delvm;
    if (delvp < phi) phi = delvp;
    if (phi < 0.f) phi = 0.f;
    if (phi > max_slope) phi = max_slope;
    return phi;
}

// EOS of one element (reference/C/LULESH-OMP.cc:2384-2561; lulesh-2.0.3/
// lulesh.cc:2043-2231): pressures, q and sound speed in float32, the energy
// and its increments in float64
struct EosConstMixed {
    double e_cut, emin, eosvmax, eosvmin;
    float p_cut, q_cut, pmin, rho0_inv, ss_tiny, ss_floor;
    bool unit_rho0;
};

struct EosOutMixed {
    double e;
    float p, q, ss;
};

__device__ __forceinline__ float eos_sound_m(float pbvc, float e, float vv, float bvc,
                                             float p, const EosConstMixed &c)
{
    float s = pbvc * e + vv * bvc * p;
    if (!c.unit_rho0) {
        s = s * c.rho0_inv;
    }
    return (s <= c.ss_tiny) ? c.ss_floor : fsqrt(s);
}

__device__ __forceinline__ float eos_pressure_m(float bvc, double e, double vnewc,
                                                const EosConstMixed &c)
{
    float p = bvc * float(e);
    if (fabsf(p) < c.p_cut) p = 0.f;
    if (vnewc >= c.eosvmax) p = 0.f;
    if (p < c.pmin) p = c.pmin;
    return p;
}

__device__ __forceinline__ EosOutMixed eos_element_mixed(double vnewc, double e_old,
                                                         float delvc, float p_old,
                                                         float q_old, float qq_old,
                                                         float ql_old,
                                                         const EosConstMixed &c)
{
    const float c1s = 2.0f / 3.0f;
    const float vn = float(vnewc);
    float compression = frcp(vn) - 1.f;
    const float vchalf = vn - delvc * .5f;
    float comp_half_step = frcp(vchalf) - 1.f;
    if (c.eosvmin != 0.) {
        if (vnewc <= c.eosvmin) comp_half_step = compression;
    }
    if (c.eosvmax != 0.) {
        if (vnewc >= c.eosvmax) {
            p_old = 0.f;
            compression = 0.f;
            comp_half_step = 0.f;
        }
    }
    const double dv = double(delvc);
    double e_new = e_old - 0.5 * dv * double(p_old + q_old);
    if (e_new < c.emin) e_new = c.emin;

    float bvc = c1s * (comp_half_step + 1.f);
    const float pbvc = c1s;
    const float p_half_step = eos_pressure_m(bvc, e_new, vnewc, c);
    const float vhalf = frcp(1.f + comp_half_step);
    float q_new;
    if (delvc > 0.f) {
        q_new = 0.f;
    } else {
        const float ssc = eos_sound_m(pbvc, float(e_new), vhalf * vhalf, bvc, p_half_step, c);
        q_new = ssc * ql_old + qq_old;
    }
    e_new = e_new + 0.5 * dv * double(3.f * (p_old + q_old) - 4.f * (p_half_step + q_new));
    if (fabs(e_new) < c.e_cut) e_new = 0.;
    if (e_new < c.emin) e_new = c.emin;

    bvc = c1s * (compression + 1.f);
    float p_new = eos_pressure_m(bvc, e_new, vnewc, c);
    {
        float q_tilde;
        if (delvc > 0.f) {
            q_tilde = 0.f;
        } else {
            const float ssc = eos_sound_m(pbvc, float(e_new), vn * vn, bvc, p_new, c);
            q_tilde = ssc * ql_old + qq_old;
        }
        e_new = e_new - double(7.f * (p_old + q_old) - 8.f * (p_half_step + q_new) +
                               (p_new + q_tilde)) *
                            dv * (1.0 / 6.0);
        if (fabs(e_new) < c.e_cut) e_new = 0.;
        if (e_new < c.emin) e_new = c.emin;
    }
    p_new = eos_pressure_m(bvc, e_new, vnewc, c);
    if (delvc <= 0.f) {
        const float ssc = eos_sound_m(pbvc, float(e_new), vn * vn, bvc, p_new, c);
        q_new = ssc * ql_old + qq_old;
        if (fabsf(q_new) < c.q_cut) q_new = 0.f;
    }
    EosOutMixed o;
    o.ss = eos_sound_m(pbvc, float(e_new), vn * vn, bvc, p_new, c);
    o.p = p_new;
    o.e = e_new;
    o.q = q_new;
    return o;
}

}  // namespace

// ---------------------------------------------------------------------------
// Kinematics and monotonic-Q gradients (reference/C/LULESH-OMP.cc:1927-2180)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_kinematics_q_mixed(DevFieldsMixed f,
                                                            DevScalars *s,
                                                            PhysParams prm)
{
    if (s->active == 0 || s->error != 0) {
        return;
    }
    const int el = int(blockIdx.x) * int(blockDim.x) + int(threadIdx.x);
    if (el >= f.num_elem) {
        return;
    }
    const int par = s->cur;
    const double dt = s->deltatime;
    int i, j, k;
    elem_ijk(f, el, i, j, k);
    const int en = f.nx + 1;
    const int n0 = (k * en + j) * en + i;
    const int pl = en * en;
    const int nodes[8] = {n0,      n0 + 1,      n0 + en + 1,      n0 + en,
                          n0 + pl, n0 + pl + 1, n0 + pl + en + 1, n0 + pl + en};
    double X[8], Y[8], Z[8], XV[8], YV[8], ZV[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        X[c] = f.x[par][nodes[c]];
        Y[c] = f.y[par][nodes[c]];
        Z[c] = f.z[par][nodes[c]];
        XV[c] = f.xd[par][nodes[c]];
        YV[c] = f.yd[par][nodes[c]];
        ZV[c] = f.zd[par][nodes[c]];
    }
    const double volo = f.volo[el];
    const double v_old = f.v[el];  // read before the stores below may alias it
    // all loads issued before any arithmetic: one wait for memory (as in
    // k_kinematics_q)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        asm volatile("" : "+v"(X[c]), "+v"(Y[c]), "+v"(Z[c]), "+v"(XV[c]), "+v"(YV[c]),
                     "+v"(ZV[c]));
    }
    __builtin_amdgcn_s_setprio(1);  // a wave with its data finishes first
    // float64: element volume, relative volume and its change
    const double volume = elem_volume(X, Y, Z);
    const double vnew = volume / volo;
    f.vnew[el] = vnew;
    f.delv[el] = float(vnew - v_old);
    if (vnew <= 0.0) {
        raise_error(s, -1);
    }
    float x[8], y[8], z[8], xv[8], yv[8], zv[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        x[c] = float(X[c] - X[0]);
        y[c] = float(Y[c] - Y[0]);
        z[c] = float(Z[c] - Z[0]);
        xv[c] = float(XV[c] - XV[0]);
        yv[c] = float(YV[c] - YV[0]);
        zv[c] = float(ZV[c] - ZV[0]);
    }
    f.arealg[el] = characteristic_length(x, y, z, float(volume));
    {
        // velocity gradient on the half-step geometry; its Jacobian in
        // float64 on coordinates relative to corner 0
        const double dt2 = 0.5 * dt;
        double xh[8], yh[8], zh[8], b[3][4];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            xh[c] = (X[c] - X[0]) - dt2 * (XV[c] - XV[0]);
            yh[c] = (Y[c] - Y[0]) - dt2 * (YV[c] - YV[0]);
            zh[c] = (Z[c] - Z[0]) - dt2 * (ZV[c] - ZV[0]);
        }
        const double inv_det_j = 1.0 / shape_derivatives(xh, yh, zh, b);
        const float dxx = float(b[0][0]) * (xv[0] - xv[6]) + float(b[0][1]) * (xv[1] - xv[7]) +
                          float(b[0][2]) * (xv[2] - xv[4]) + float(b[0][3]) * (xv[3] - xv[5]);
        const float dyy = float(b[1][0]) * (yv[0] - yv[6]) + float(b[1][1]) * (yv[1] - yv[7]) +
                          float(b[1][2]) * (yv[2] - yv[4]) + float(b[1][3]) * (yv[3] - yv[5]);
        const float dzz = float(b[2][0]) * (zv[0] - zv[6]) + float(b[2][1]) * (zv[1] - zv[7]) +
                          float(b[2][2]) * (zv[2] - zv[4]) + float(b[2][3]) * (zv[3] - zv[5]);
        f.vdov[el] = float(inv_det_j * double(dxx + dyy + dzz));
    }

    // monotonic-Q gradients, float32
    const float ptiny = 1.e-36f;
    const float vol = float(volo * vnew);
    const float norm = frcp(vol + ptiny);
    const float dxj = -0.25f * ((x[0] + x[1] + x[5] + x[4]) - (x[3] + x[2] + x[6] + x[7]));
    const float dyj = -0.25f * ((y[0] + y[1] + y[5] + y[4]) - (y[3] + y[2] + y[6] + y[7]));
    const float dzj = -0.25f * ((z[0] + z[1] + z[5] + z[4]) - (z[3] + z[2] + z[6] + z[7]));
    const float dxi = 0.25f * ((x[1] + x[2] + x[6] + x[5]) - (x[0] + x[3] + x[7] + x[4]));
    const float dyi = 0.25f * ((y[1] + y[2] + y[6] + y[5]) - (y[0] + y[3] + y[7] + y[4]));
    const float dzi = 0.25f * ((z[1] + z[2] + z[6] + z[5]) - (z[0] + z[3] + z[7] + z[4]));
    const float dxk = 0.25f * ((x[4] + x[5] + x[6] + x[7]) - (x[0] + x[1] + x[2] + x[3]));
    const float dyk = 0.25f * ((y[4] + y[5] + y[6] + y[7]) - (y[0] + y[1] + y[2] + y[3]));
    const float dzk = 0.25f * ((z[4] + z[5] + z[6] + z[7]) - (z[0] + z[1] + z[2] + z[3]));
    float ax, ay, az, dxv, dyv, dzv;

    ax = dyi * dzj - dzi * dyj;
    ay = dzi * dxj - dxi * dzj;
    az = dxi * dyj - dyi * dxj;
    f.delx_zeta[el] = vol * frsq(ax * ax + ay * ay + az * az + ptiny);
    ax *= norm;
    ay *= norm;
    az *= norm;
    dxv = 0.25f * ((xv[4] + xv[5] + xv[6] + xv[7]) - (xv[0] + xv[1] + xv[2] + xv[3]));
    dyv = 0.25f * ((yv[4] + yv[5] + yv[6] + yv[7]) - (yv[0] + yv[1] + yv[2] + yv[3]));
    dzv = 0.25f * ((zv[4] + zv[5] + zv[6] + zv[7]) - (zv[0] + zv[1] + zv[2] + zv[3]));
    f.delv_zeta[el] = ax * dxv + ay * dyv + az * dzv;

    ax = dyj * dzk - dzj * dyk;
    ay = dzj * dxk - dxj * dzk;
    az = dxj * dyk - dyj * dxk;
    f.delx_xi[el] = vol * frsq(ax * ax + ay * ay + az * az + ptiny);
    ax *= norm;
    ay *= norm;
    az *= norm;
    dxv = 0.25f * ((xv[1] + xv[2] + xv[6] + xv[5]) - (xv[0] + xv[3] + xv[7] + xv[4]));
    dyv = 0.25f * ((yv[1] + yv[2] + yv[6] + yv[5]) - (yv[0] + yv[3] + yv[7] + yv[4]));
    dzv = 0.25f * ((zv[1] + zv[2] + zv[6] + zv[5]) - (zv[0] + zv[3] + zv[7] + zv[4]));
    f.delv_xi[el] = ax * dxv + ay * dyv + az * dzv;

    ax = dyk * dzi - dzk * dyi;
    ay = dzk * dxi - dxk * dzi;
    az = dxk * dyi - dyk * dxi;
    f.delx_eta[el] = vol * frsq(ax * ax + ay * ay + az * az + ptiny);
    ax *= norm;
    ay *= norm;
    az *= norm;
    dxv = -0.25f * ((xv[0] + xv[1] + xv[5] + xv[4]) - (xv[3] + xv[2] + xv[6] + xv[7]));
    dyv = -0.25f * ((yv[0] + yv[1] + yv[5] + yv[4]) - (yv[3] + yv[2] + yv[6] + yv[7]));
    dzv = -0.25f * ((zv[0] + zv[1] + zv[5] + zv[4]) - (zv[3] + zv[2] + zv[6] + zv[7]));
    f.delv_eta[el] = ax * dxv + ay * dyv + az * dzv;
}

// ---------------------------------------------------------------------------
// Monotonic Q, EOS, volume update and time constraints; the structure of
// k_q_eos_dt and k_q_eos_dt_nat (lulesh_kernels.hip)
// ---------------------------------------------------------------------------
namespace {

struct EosInMixed {
    double vnewc, e_old;
    float delvc, p_old, q_old, qquad, qlin;
};

// what an element keeps for its stores after the EOS
struct QKeepMixed {
    double vnew;
    float vdov, arealg;
};

__device__ __forceinline__ EosConstMixed eos_const_mixed(const PhysParams &prm)
{
    EosConstMixed ec;
    ec.e_cut = prm.e_cut;
    ec.emin = prm.emin;
    ec.eosvmax = prm.eosvmax;
    ec.eosvmin = prm.eosvmin;
    ec.p_cut = float(prm.p_cut);
    ec.q_cut = float(prm.q_cut);
    ec.pmin = float(prm.pmin);
    ec.rho0_inv = float(1.0 / prm.refdens);
    ec.unit_rho0 = prm.refdens == 1.0;
    ec.ss_tiny = float(prm.ss_tiny);
    ec.ss_floor = float(prm.ss_floor);
    return ec;
}

// The element's monotonic Q (ql / qq stored) and its side of the EOS before
// the evaluations: qstop tested on the previous cycle's q, the new and old
// relative volumes clamped and the clamped old volume tested
// (reference/C/LULESH-OMP.cc:2183-2320, :2368-2381; lulesh-2.0.3/
// lulesh.cc:2704-2753).  The element's inputs are all loaded before its
// first store.
__device__ __forceinline__ EosInMixed q_eos_prepare_mixed(const DevFieldsMixed &f,
                                                          DevScalars *s, const PhysParams &prm,
                                                          int el, QKeepMixed &kp)
{
    const int nx = f.nx;
    int i, j, k;
    elem_ijk(f, el, i, j, k);
    const int sy = nx, sz = nx * nx;

    const float dvxi = f.delv_xi[el], dveta = f.delv_eta[el], dvzeta = f.delv_zeta[el];
    // neighbours across a boundary face come from the element itself and
    // are then replaced
    const float xm = f.delv_xi[(i == 0) ? el : el - 1];
    const float xp = f.delv_xi[(i == nx - 1) ? el : el + 1];
    const float ym = f.delv_eta[(j == 0) ? el : el - sy];
    const float yp = f.delv_eta[(j == nx - 1) ? el : el + sy];
    const float zm = f.delv_zeta[(k == 0) ? el : el - sz];
    const float zp = f.delv_zeta[(k == nx - 1) ? el : el + sz];
    const float vdov = f.vdov[el];
    const double vnew = f.vnew[el];
    const double volo = f.volo[el];
    const float q_old = f.q[el];
    const double v_old = f.v[el];
    const double e_old = f.e[el];
    const float delvc = f.delv[el], p_old = f.p[el];
    const float arealg = (vdov != 0.f) ? f.arealg[el] : 0.f;
    const float lm = float(prm.monoq_limiter_mult), ms = float(prm.monoq_max_slope);
    const float phixi = mono_phi(dvxi, (i == 0) ? dvxi : xm, (i == nx - 1) ? 0.f : xp, lm, ms);
    const float phieta = mono_phi(dveta, (j == 0) ? dveta : ym, (j == nx - 1) ? 0.f : yp, lm, ms);
    const float phizeta =
        mono_phi(dvzeta, (k == 0) ? dvzeta : zm, (k == nx - 1) ? 0.f : zp, lm, ms);
    float qlin, qquad;
    if (vdov > 0.f) {
        qlin = 0.f;
        qquad = 0.f;
    } else {
        float dxi = dvxi * f.delx_xi[el];
        float deta = dveta * f.delx_eta[el];
        float dzeta = dvzeta * f.delx_zeta[el];
        if (dxi > 0.f) dxi = 0.f;
        if (deta > 0.f) deta = 0.f;
        if (dzeta > 0.f) dzeta = 0.f;
        const float rho = float(f.elem_mass[el]) * frcp(float(volo * vnew));
        qlin = -float(prm.qlc_monoq) * rho *
               (dxi * (1.f - phixi) + deta * (1.f - phieta) + dzeta * (1.f - phizeta));
        qquad = float(prm.qqc_monoq) * rho *
                (dxi * dxi * (1.f - phixi * phixi) + deta * deta * (1.f - phieta * phieta) +
                 dzeta * dzeta * (1.f - phizeta * phizeta));
    }
    f.ql[el] = qlin;
    f.qq[el] = qquad;

    if (double(q_old) > prm.qstop) {
        raise_error(s, -2);
    }
    double vnewc = vnew;
    if (prm.eosvmin != 0.) {
        if (vnewc < prm.eosvmin) vnewc = prm.eosvmin;
    }
    if (prm.eosvmax != 0.) {
        if (vnewc > prm.eosvmax) vnewc = prm.eosvmax;
    }
    double vc = v_old;
    if (prm.eosvmin != 0.) {
        if (vc < prm.eosvmin) vc = prm.eosvmin;
    }
    if (prm.eosvmax != 0.) {
        if (vc > prm.eosvmax) vc = prm.eosvmax;
    }
    if (vc <= 0.) {
        raise_error(s, -1);
    }
    kp.vnew = vnew;
    kp.vdov = vdov;
    kp.arealg = arealg;
    return EosInMixed{vnewc, e_old, delvc, p_old, q_old, qquad, qlin};
}

// `rep` evaluations of the EOS on the same inputs, as the reference repeats
// them (lulesh-2.0.3/lulesh.cc:2413-2424): the inputs pass through an empty
// asm statement at the top of every repetition, carried in the same
// registers, so each repetition is computed in full, and every result is
// marked as used.
__device__ __forceinline__ EosOutMixed eos_repeat_mixed(const EosInMixed &a, int rep,
                                                        const EosConstMixed &ec)
{
    double a0 = a.vnewc, a1 = a.e_old;
    float a2 = a.delvc, a3 = a.p_old, a4 = a.q_old, a5 = a.qquad, a6 = a.qlin;
    EosOutMixed o;
    o.e = 0.0;
    o.p = o.q = o.ss = 0.f;
    for (int r = 0; r < rep; ++r) {
        asm volatile("" : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5),
                     "+v"(a6));
        o = eos_element_mixed(a0, a1, a2, a3, a4, a5, a6, ec);
        asm volatile("" ::"v"(o.p), "v"(o.e), "v"(o.q), "v"(o.ss));
    }
    return o;
}

// The element's side after the EOS: p, e, q, ss stored, the volume update
// (1.0 keeps the unclamped vnew, 2.0 the clamped one, lulesh-2.0.3/
// lulesh.cc:2439-2452) and the Courant and hydro candidates (:2799-2933).
__device__ __forceinline__ void eos_finish_mixed(const DevFieldsMixed &f,
                                                 const PhysParams &prm, int el,
                                                 const QKeepMixed &kp, double vnewc,
                                                 const EosOutMixed &o,
                                                 unsigned long long &cand_c,
                                                 unsigned long long &cand_h)
{
    f.p[el] = o.p;
    f.e[el] = o.e;
    f.q[el] = o.q;
    f.ss[el] = o.ss;
    double tmpv = (prm.ic_mode == 1) ? kp.vnew : vnewc;
    if (fabs(tmpv - 1.0) < prm.v_cut) tmpv = 1.0;
    f.v[el] = tmpv;
    if (prm.ic_mode == 2) {
        f.vnew[el] = vnewc;
    }
    const float vdov = kp.vdov;
    if (vdov != 0.f) {
        const float qqc2 = float(64.0 * prm.qqc * prm.qqc);
        float dtf = o.ss * o.ss;
        if (vdov < 0.f) {
            dtf = dtf + qqc2 * kp.arealg * kp.arealg * vdov * vdov;
        }
        cand_c = as_bits(double(kp.arealg * frsq(dtf)));
        cand_h = as_bits(prm.dvovmax / (double(fabsf(vdov)) + 1.e-20));
    }
}

__device__ __forceinline__ void fold_minima_mixed(DevScalars *s, unsigned long long cand_c,
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

// Per block: the EOS inputs of the elements with more than one evaluation,
// by place, and each wave's counts (ExtraDeal).
struct RepLdsMixed {
    double in_d[2][256];
    float in_f[5][256];
    int cnt[4];
};

// The EOS evaluations of a block's elements beyond each one's first, dealt
// out over all 256 threads (the scheme of eos_extra_evaluations in
// lulesh_kernels.hip): the thread that owns an element evaluates it once and
// keeps that result; the others take ceil(sum(rep - 1) / 256) passes of the
// block.  Each is computed in full and its result marked as used.  Every
// thread of the block calls it.
__device__ __forceinline__ void eos_extra_evaluations_mixed(const EosInMixed &a, int extra,
                                                            const int (&classes)[2],
                                                            const EosConstMixed &ec,
                                                            RepLdsMixed &L)
{
    const ExtraDeal deal(extra, classes, L.cnt);
    if (deal.total == 0) {  // the same for every thread of the block
        return;
    }
    if (deal.place >= 0) {
        L.in_d[0][deal.place] = a.vnewc;
        L.in_d[1][deal.place] = a.e_old;
        L.in_f[0][deal.place] = a.delvc;
        L.in_f[1][deal.place] = a.p_old;
        L.in_f[2][deal.place] = a.q_old;
        L.in_f[3][deal.place] = a.qquad;
        L.in_f[4][deal.place] = a.qlin;
    }
    __syncthreads();
    for (int w = int(threadIdx.x); w < deal.total; w += 256) {
        const int src = deal.owner(w);
        double b0 = L.in_d[0][src], b1 = L.in_d[1][src];
        float b2 = L.in_f[0][src], b3 = L.in_f[1][src], b4 = L.in_f[2][src];
        float b5 = L.in_f[3][src], b6 = L.in_f[4][src];
        asm volatile("" : "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3), "+v"(b4), "+v"(b5),
                     "+v"(b6));
        const EosOutMixed o = eos_element_mixed(b0, b1, b2, b3, b4, b5, b6, ec);
        asm volatile("" ::"v"(o.p), "v"(o.e), "v"(o.q), "v"(o.ss));
    }
}

}  // namespace

// The region-ordered schedule: block b takes chunk eos_chunk(b) of the
// elements sorted by region, each thread running its element's repetitions.
__global__ __launch_bounds__(256) void k_q_eos_dt_mixed(DevFieldsMixed f, DevScalars *s,
                                                        PhysParams prm, int bands)
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
    const int slot = eos_chunk(int(blockIdx.x), int(gridDim.x), bands) * int(blockDim.x) +
                     int(threadIdx.x);
    __builtin_amdgcn_s_setprio(1);  // the element's loads first
    unsigned long long cand_c = as_bits(kBig), cand_h = as_bits(kBig);
    if (slot < f.num_elem) {
        const int el = f.eos_order[slot];
        const int rep = f.eos_rep[slot];
        QKeepMixed kp;
        const EosInMixed a = q_eos_prepare_mixed(f, s, prm, el, kp);
        const EosConstMixed ec = eos_const_mixed(prm);
        __builtin_amdgcn_s_setprio(0);  // the repetitions yield to waves still loading
        const EosOutMixed o = eos_repeat_mixed(a, rep, ec);
        __builtin_amdgcn_s_setprio(1);  // stores and the block's reduction
        eos_finish_mixed(f, prm, el, kp, a.vnewc, o, cand_c, cand_h);
    }
    fold_minima_mixed(s, cand_c, cand_h, lds_c, lds_h);
}

// Mesh order, one element per thread, blocks of f.eos_elems consecutive elements in
// the order f.eos_blocks gives, the regions' EOS repetitions shared over
// each block's threads (as k_q_eos_dt_nat).  Each element's arithmetic is
// that of k_q_eos_dt_mixed, so both give the same bits.
__global__ __launch_bounds__(256) void k_q_eos_dt_mixed_nat(DevFieldsMixed f, DevScalars *s,
                                                            PhysParams prm)
{
    __shared__ unsigned long long lds_c[4], lds_h[4];
    __shared__ int skip;
    __shared__ RepLdsMixed rep_lds;
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
    const EosConstMixed ec = eos_const_mixed(prm);
    unsigned long long cand_c = as_bits(kBig), cand_h = as_bits(kBig);
    QKeepMixed kp{1.0, 0.f, 0.f};
    EosInMixed a{1.0, 0.0, 0.f, 0.f, 0.f, 0.f, 0.f};
    int extra = 0;
    if (valid) {
        extra = int(f.rep[el]) - 1;
        a = q_eos_prepare_mixed(f, s, prm, el, kp);
    }
    __builtin_amdgcn_s_setprio(0);  // the evaluations yield to waves still loading
    const EosOutMixed o = eos_repeat_mixed(a, 1, ec);
    eos_extra_evaluations_mixed(a, extra, f.eos_extra, ec, rep_lds);
    __builtin_amdgcn_s_setprio(1);  // stores and the block's reduction
    if (valid) {
        eos_finish_mixed(f, prm, el, kp, a.vnewc, o, cand_c, cand_h);
    }
    fold_minima_mixed(s, cand_c, cand_h, lds_c, lds_h);
}

#define LULESH_MIXED_SHAPES(X) \
    X(32, 8, 2)                \
    X(32, 8, 3)                \
    X(16, 16, 3)               \
    X(16, 8, 3)                \
    X(32, 16, 2)

bool force_sweep_mixed_shape_supported(const SweepShape &sh)
{
    if (sh.nz < 1 || sh.nz > 4096) {
        return false;
    }
#define LULESH_MATCH(a, b, w) \
    if (sh.tx == a && sh.ty == b && sh.waves == w) return true;
    LULESH_MIXED_SHAPES(LULESH_MATCH)
#undef LULESH_MATCH
    return false;
}

hipError_t launch_force_sweep_mixed(const SweepShape &sh, const DevFieldsMixed &f,
                                    const DevScalars *from, DevScalars *s,
                                    const PhysParams &prm, hipStream_t stream)
{
    if (sh.nz < 1) {
        return hipErrorInvalidValue;
    }
#define LULESH_LAUNCH(a, b, w)                     \
    if (sh.tx == a && sh.ty == b && sh.waves == w) \
        return launch_mixed_shape<a, b, w>(sh.nz, f, from, s, prm, stream);
    LULESH_MIXED_SHAPES(LULESH_LAUNCH)
#undef LULESH_LAUNCH
    return hipErrorInvalidValue;
}

}  // namespace lulesh
