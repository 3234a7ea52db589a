// hd_fused.h -- what the fused kernels share: the basis and quadrature rules as
// compile-time constants, face polynomials, mode loads, the limiter; and the
// 13-moment cell kernel of the table-driven path.
//
// Operator (the reference's glflux + innerintegral2 + source_calc +
// advance_time_level, src/flux.f90:751-1022, src/sources.f90:12-84,
// src/integrator.f90:125-252), with dQ/dt = -glflux + source:
//   RHS[f][r] = sum_d dxi_d * ( sum_g Cvol(d,r,g) F_d(Q(g))[f]
//                             + sum_p Cface(-d,r,p) Fhat_{-d}(p)[f]
//                             + sum_p Cface(+d,r,p) Fhat_{+d}(p)[f] )  + source
//   Cvol  = 0.25 cb_r w3_g dphi_r/dxi_d(g),  Cface(-d) = +0.25 cb_r w2_p phi_r(-d,p),
//   Cface(+d) = -0.25 cb_r w2_p phi_r(+d,p).
// The basis is the Legendre product of src/basis_funcs.f90 with the mode order
// of src/initialize.f90:126-194; quadrature nodes and weights are the
// reference's values (1/sqrt(3); sqrt(15)/5, 5/9, 8/9) as exact hex literals.
#pragma once
#include "hd_generic.h"
#include "hd_prim.h"

namespace hd {
namespace fz {

// ---------------------------------------------------------------- rules ----
template <int QP>
struct Rule;
template <>
struct Rule<2> {
    static HD_DEV constexpr double x(int i) { return i == 0 ? -0x1.279a74590331dp-1 : 0x1.279a74590331dp-1; }
    static HD_DEV constexpr double w(int) { return 1.0; }
    static HD_DEV constexpr double p2(int) { return 0x1.0p-53; }  // 1.5*s*s - 0.5 at s = 1/sqrt(3)
    static HD_DEV constexpr double w2(int, int) { return 1.0; }
    static HD_DEV constexpr double w3(int, int, int) { return 1.0; }
};
template <>
struct Rule<3> {
    static HD_DEV constexpr double x(int i) {
        return i == 0 ? -0x1.8c97ef43f7248p-1 : (i == 1 ? 0.0 : 0x1.8c97ef43f7248p-1);
    }
    static HD_DEV constexpr double w(int i) { return i == 1 ? 0x1.c71c71c71c71cp-1 : 0x1.1c71c71c71c72p-1; }
    static HD_DEV constexpr double p2(int i) { return i == 1 ? -0.5 : 0x1.999999999999cp-2; }
    // set_weights_3D: w2(i,j) = w1(j)*w1(i); w3(i; j,k) = w2(j,k)*w1(i)
    static HD_DEV constexpr double w2(int i, int j) { return w(j) * w(i); }
    static HD_DEV constexpr double w3(int i, int j, int k) { return w2(j, k) * w(i); }
};

// ---------------------------------------------------------------- basis ----
// Legendre degrees (a,b,c) in (x,y,z) of mode r
template <int NB>
HD_DEV constexpr int deg(int r, int ax) {
    // 1, x, y, z, yz, zx, xy, then xyz (NB 8) or P2x, P2y, P2z (NB 10); pure
    // arithmetic so that no lookup array is ever materialised on the device
    return r == 0 ? 0
         : r <= 3 ? (ax == r - 1 ? 1 : 0)
         : r <= 6 ? (ax == r - 4 ? 0 : 1)
         : (NB == 8 ? 1 : (ax == r - 7 ? 2 : 0));
}
template <int NB>
HD_DEV constexpr double cbasis(int r) {
    return double((2 * deg<NB>(r, 0) + 1) * (2 * deg<NB>(r, 1) + 1) * (2 * deg<NB>(r, 2) + 1));
}
template <int QP>
HD_DEV constexpr double Lval(int a, int i) { return a == 0 ? 1.0 : (a == 1 ? Rule<QP>::x(i) : Rule<QP>::p2(i)); }
// value at the face where the coordinate is -1 (side 0) or +1 (side 1)
HD_DEV constexpr double Lface(int a, int side) { return a == 1 ? (side ? 1.0 : -1.0) : 1.0; }
template <int QP>
HD_DEV constexpr double Dval(int a, int i) { return a == 0 ? 0.0 : (a == 1 ? 1.0 : 3.0 * Rule<QP>::x(i)); }

// interior point g = (i,j,k), x index slowest
template <int NB, int QP>
HD_DEV constexpr double phi_int(int r, int i, int j, int k) {
    return Lval<QP>(deg<NB>(r, 0), i) * Lval<QP>(deg<NB>(r, 1), j) * Lval<QP>(deg<NB>(r, 2), k);
}
// 0.25*cb_r*w3_g*d(phi_r)/d(xi_d) at g
template <int NB, int QP>
HD_DEV constexpr double cvol(int d, int r, int i, int j, int k) {
    const double a = d == 0 ? Dval<QP>(deg<NB>(r, 0), i) : Lval<QP>(deg<NB>(r, 0), i);
    const double b = d == 1 ? Dval<QP>(deg<NB>(r, 1), j) : Lval<QP>(deg<NB>(r, 1), j);
    const double c = d == 2 ? Dval<QP>(deg<NB>(r, 2), k) : Lval<QP>(deg<NB>(r, 2), k);
    return 0.25 * cbasis<NB>(r) * Rule<QP>::w3(i, j, k) * (a * b * c);
}
// d(phi_r)/d(xi_d) at g
template <int NB, int QP>
HD_DEV constexpr double dphi(int d, int r, int i, int j, int k) {
    const double a = d == 0 ? Dval<QP>(deg<NB>(r, 0), i) : Lval<QP>(deg<NB>(r, 0), i);
    const double b = d == 1 ? Dval<QP>(deg<NB>(r, 1), j) : Lval<QP>(deg<NB>(r, 1), j);
    const double c = d == 2 ? Dval<QP>(deg<NB>(r, 2), k) : Lval<QP>(deg<NB>(r, 2), k);
    return a * b * c;
}
// face point p = (ii,jj), jj fastest: x faces (y=x[jj], z=x[ii]); y faces
// (x=x[ii], z=x[jj]); z faces (x=x[jj], y=x[ii])  (src/basis_funcs.f90:346-567)
template <int NB, int QP>
HD_DEV constexpr double phi_face(int dir, int side, int r, int ii, int jj) {
    const int a = deg<NB>(r, 0), b = deg<NB>(r, 1), c = deg<NB>(r, 2);
    if (dir == 0) return Lface(a, side) * Lval<QP>(b, jj) * Lval<QP>(c, ii);
    if (dir == 1) return Lval<QP>(a, ii) * Lface(b, side) * Lval<QP>(c, jj);
    return Lval<QP>(a, jj) * Lval<QP>(b, ii) * Lface(c, side);
}
template <int NB, int QP>
HD_DEV constexpr double cface(int dir, int side, int r, int ii, int jj) {
    return (side ? -0.25 : 0.25) * cbasis<NB>(r) * Rule<QP>::w2(ii, jj) * phi_face<NB, QP>(dir, side, r, ii, jj);
}

// Face tables in constant memory for the runtime point loops:
//   bf[dir][side][p][r] = phi_r on that face at point p
//   cf[dir][side][p][r] = cface
template <int NB, int QP>
struct FaceTab {
    double bf[3][2][QP * QP][NB];
    double cf[3][2][QP * QP][NB];
};
template <int NB, int QP>
constexpr FaceTab<NB, QP> make_face_tab() {
    FaceTab<NB, QP> t{};
    for (int d = 0; d < 3; d++)
        for (int s = 0; s < 2; s++)
            for (int ii = 0; ii < QP; ii++)
                for (int jj = 0; jj < QP; jj++)
                    for (int r = 0; r < NB; r++) {
                        t.bf[d][s][ii * QP + jj][r] = phi_face<NB, QP>(d, s, r, ii, jj);
                        t.cf[d][s][ii * QP + jj][r] = cface<NB, QP>(d, s, r, ii, jj);
                    }
    return t;
}
static __constant__ FaceTab<4, 2> c_face_4 = make_face_tab<4, 2>();
static __constant__ FaceTab<8, 2> c_face_8 = make_face_tab<8, 2>();
static __constant__ FaceTab<10, 3> c_face_10 = make_face_tab<10, 3>();
template <int NB>
__device__ __forceinline__ const FaceTab<NB, (NB == 10 ? 3 : 2)>& face_tab();
template <>
__device__ __forceinline__ const FaceTab<4, 2>& face_tab<4>() { return c_face_4; }
template <>
__device__ __forceinline__ const FaceTab<8, 2>& face_tab<8>() { return c_face_8; }
template <>
__device__ __forceinline__ const FaceTab<10, 3>& face_tab<10>() { return c_face_10; }

// ------------------------------------------------------ face traces ------
// On a face the basis collapses to a polynomial in the two tangential
// coordinates (row = the ii coordinate, col = the jj coordinate of the face
// point order above): phi_r = Lface(normal degree) * L(dr, row) * L(dc, col),
// with (dr, dc) in {(0,0), (1,0), (0,1), (1,1), (2,0), (0,2)}.  A side's
// trace is therefore sum_k K_k b_k(p) with NK = 3 (nb 4), 4 (nb 8) or 6
// (nb 10) coefficients K_k = sum of +-m_r over the modes of pair k: NK
// products per point instead of NB.  Coefficients and values come from
// sg::signed_coeffs and sg::eval_point everywhere, so that all that evaluate a
// side's trace agree bitwise.
template <int NB>
HD_DEV constexpr int face_nk() { return NB == 10 ? 6 : (NB == 8 ? 4 : 3); }
HD_DEV constexpr int pair_index(int dr, int dc) {
    return dr == 0 ? (dc == 0 ? 0 : (dc == 1 ? 2 : 5)) : (dr == 1 ? (dc == 0 ? 1 : 3) : 4);
}
HD_DEV constexpr int pair_dr(int k) { return k == 1 || k == 3 ? 1 : (k == 4 ? 2 : 0); }
HD_DEV constexpr int pair_dc(int k) { return k == 2 || k == 3 ? 1 : (k == 5 ? 2 : 0); }
// tangential axes of a face: row = ii coordinate, col = jj coordinate
HD_DEV constexpr int row_axis(int dir) { return dir == 0 ? 2 : (dir == 1 ? 0 : 1); }
HD_DEV constexpr int col_axis(int dir) { return dir == 0 ? 1 : (dir == 1 ? 2 : 0); }

// b_k at face point p = (ii, jj), jj fastest, and w2_p*b_k (lifts)
template <int NB, int QP>
struct FacePoly {
    double b[QP * QP][face_nk<NB>()];
    double wb[QP * QP][face_nk<NB>()];
};
template <int NB, int QP>
constexpr FacePoly<NB, QP> make_face_poly() {
    FacePoly<NB, QP> t{};
    for (int ii = 0; ii < QP; ii++)
        for (int jj = 0; jj < QP; jj++)
            for (int k = 0; k < face_nk<NB>(); k++) {
                t.b[ii * QP + jj][k] = Lval<QP>(pair_dr(k), ii) * Lval<QP>(pair_dc(k), jj);
                t.wb[ii * QP + jj][k] = Rule<QP>::w2(ii, jj) * t.b[ii * QP + jj][k];
            }
    return t;
}
static __constant__ FacePoly<4, 2> c_fpoly_4 = make_face_poly<4, 2>();
static __constant__ FacePoly<8, 2> c_fpoly_8 = make_face_poly<8, 2>();
static __constant__ FacePoly<10, 3> c_fpoly_10 = make_face_poly<10, 3>();
template <int NB>
__device__ __forceinline__ const FacePoly<NB, (NB == 10 ? 3 : 2)>& face_poly();
template <>
__device__ __forceinline__ const FacePoly<4, 2>& face_poly<4>() { return c_fpoly_4; }
template <>
__device__ __forceinline__ const FacePoly<8, 2>& face_poly<8>() { return c_fpoly_8; }
template <>
__device__ __forceinline__ const FacePoly<10, 3>& face_poly<10>() { return c_fpoly_10; }

// Keeps the scheduler from interleaving fully unrolled quadrature points,
// which would stretch live ranges past the register file.
__device__ __forceinline__ void point_barrier() { __builtin_amdgcn_sched_barrier(0); }

// ------------------------------------------------------------- faces -------
struct CellPos {
    int i, j, k;
    long c;
};

// The planes are reached by stepping one pointer a plane at a time; the
// empty asm hides the step count from the compiler, which would otherwise
// keep all NB*NQ plane offsets live in scalar registers (and spill them).
template <int NB, int NQ>
__device__ __forceinline__ void load_modes(const double* __restrict__ q, long N, long c, double (&m)[NQ][NB]) {
    // a global (address space 1) pointer, so the loads stay global loads
    const __attribute__((address_space(1))) double* p = (const __attribute__((address_space(1))) double*)(q + c);
#pragma unroll
    for (int r = 0; r < NB; r++)
#pragma unroll
        for (int f = 0; f < NQ; f++) {
            m[f][r] = *p;
            p += N;
            asm volatile("" : "+v"(p));
        }
}
template <int NB, int NQ>
__device__ __forceinline__ void load_modes(const double* __restrict__ q, const Grid& g, long c, double (&m)[NQ][NB]) {
    load_modes<NB, NQ>(q, g.N, c, m);
}

// Exterior state of an x-low inflow face point: inflow holds the reference's
// Qxlo_ext_def(ny,nz,nface,nQ) in Fortran order.
template <int NQ>
__device__ __forceinline__ void inflow_ghost(const double* __restrict__ inflow, const Grid& g, const CellPos& cp,
                                             int p, int nface, double* oth) {
    const long plane = (long)g.ny * g.nz;
    const long base = (long)cp.j + (long)g.ny * cp.k + plane * p;
    const long fs = plane * nface;  // stride of one field
    oth[RH] = inflow[base + fs * RH];
    oth[MX] = inflow[base + fs * MX];
    oth[MY] = 0.0;
    oth[MZ] = 0.0;
    oth[EN] = inflow[base + fs * EN];
}

// ----------------------------------------------------------- limiter -------
// limiter (src/flux.f90:1077-1164), in place, compile-time face tables.  The
// pressure step takes the minimum face pressure first and divides once:
// (Pave-epsP)/(Pave-P) is monotone in P for P < epsP <= Pave, so this equals
// the reference's minimum over points.
// Exact early-out.  Every basis function is bounded by 1 in magnitude at the
// face points (products of L0 = 1, L1 and L2 on [-1,1]), so
// rho(p) >= rho_1 - sum_{r>1} |rho_r|, E(p) >= E_1 - sum |E_r|,
// |m(p)|^2 <= sum_a (sum_r |m_a,r|)^2, and the face pressure is bounded below
// by gm1*(E_lb - |m|^2_ub/(2 rho_lb)).  When both bounds clear the floors (with
// a relative margin far above rounding), the limiter's minima clear them too
// and it leaves the cell unchanged, so its face loops can be skipped.
template <int NB, int MQ>
__device__ __forceinline__ bool limiter_inactive(const double (&m)[MQ][NB], const LimParams& lp) {
    double sr = 0., se = 0., mm[3] = {0., 0., 0.};
#pragma unroll
    for (int r = 1; r < NB; r++) {
        sr += fabs(m[RH][r]);
        se += fabs(m[EN][r]);
#pragma unroll
        for (int a = 0; a < 3; a++) mm[a] += fabs(m[MX + a][r]);
    }
    const double rlb = m[RH][0] - sr;
    if (!(rlb > lp.rh_floor + 1e-10 * (fabs(m[RH][0]) + sr))) return false;
    double m2 = 0.;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double b = fabs(m[MX + a][0]) + mm[a];
        m2 += b * b;
    }
    const double Pave =
        lp.gm1 * (m[EN][0] - 0.5 * (m[MX][0] * m[MX][0] + m[MY][0] * m[MY][0] + m[MZ][0] * m[MZ][0]) / m[RH][0]);
    if (Pave < lp.epsP) return false;
    const double kin = 0.5 * m2 / rlb;
    const double plb = lp.gm1 * (m[EN][0] - se - kin);
    return plb > lp.epsP + 1e-10 * lp.gm1 * (fabs(m[EN][0]) + se + kin);
}

// Limits the modes m[0..4][*] of one cell in place; returns true if changed.
template <int NB, int QP, int MQ>
__device__ __forceinline__ bool limit_cell(double (&m)[MQ][NB], const LimParams& lp) {
    bool changed = false;
    if (m[RH][0] < lp.rh_floor) {
#pragma unroll
        for (int r = 1; r < NB; r++)
#pragma unroll
            for (int f = 0; f < 5; f++) m[f][r] = 0.0;
        m[RH][0] = lp.rh_floor;
        changed = true;
    } else if (limiter_inactive<NB, MQ>(m, lp)) {
        // no face point can reach a floor: the loops below would change nothing
    } else {
        const auto& T = face_tab<NB>();
        double rmin = 0.;
#pragma unroll 1
        for (int p = 0; p < 6 * QP * QP; p++) {
            const double* b = T.bf[p / (2 * QP * QP)][(p / (QP * QP)) % 2][p % (QP * QP)];
            double s = 0.;
#pragma unroll
            for (int r = 0; r < NB; r++) s += b[r] * m[RH][r];
            rmin = (p == 0) ? s : (s < rmin ? s : rmin);
        }
        if (rmin < lp.rh_floor) {
            double theta = (lp.rh_floor - m[RH][0]) / (rmin - m[RH][0]);
            if (theta > 1.) theta = 1.;
            if (theta < 0.) theta = 0.;
#pragma unroll
            for (int r = 1; r < NB; r++) m[RH][r] = fabs(theta) * m[RH][r];
            changed = true;
        }
        const double Pave =
            lp.gm1 * (m[EN][0] - 0.5 * (m[MX][0] * m[MX][0] + m[MY][0] * m[MY][0] + m[MZ][0] * m[MZ][0]) / m[RH][0]);
        if (Pave < lp.epsP) {
#pragma unroll
            for (int r = 1; r < NB; r++)
#pragma unroll
                for (int f = 0; f < 5; f++) m[f][r] = 0.0;
            changed = true;
        } else {
            double pmin = 0.;
#pragma unroll 1
            for (int p = 0; p < 6 * QP * QP; p++) {
                const double* b = T.bf[p / (2 * QP * QP)][(p / (QP * QP)) % 2][p % (QP * QP)];
                double e[5];
#pragma unroll
                for (int f = 0; f < 5; f++) {
                    double s = 0.;
#pragma unroll
                    for (int r = 0; r < NB; r++) s += b[r] * m[f][r];
                    e[f] = s;
                }
                const double dni = pr::rcp(e[RH]);
                const double P = lp.gm1 * (e[EN] - 0.5 * dni * (e[MX] * e[MX] + e[MY] * e[MY] + e[MZ] * e[MZ]));
                pmin = (p == 0) ? P : (P < pmin ? P : pmin);
            }
            if (pmin < lp.epsP && Pave != pmin) {
                double theta = (Pave - lp.epsP) / (Pave - pmin);
                if (theta > 1.) theta = 1.;
                if (theta < 0.) theta = 0.;
                if (theta != 1.) {
#pragma unroll
                    for (int r = 1; r < NB; r++)
#pragma unroll
                        for (int f = 0; f < 5; f++) m[f][r] = theta * m[f][r];
                    changed = true;
                }
            }
        }
    }
    return changed;
}

// get_min_dt and the limiter of a step's first stage in one pass: the wave
// speeds of the cells as they come, their modes as the limiter leaves them.
// For grids whose step is bound by its launches.  One block stores dt itself;
// several leave their maxima and, after them, the last cell's sound speed in
// partial, for k_dt_finish.
template <int NB, int QP>
__global__ __launch_bounds__(256, (NB == 4 ? 4 : (NB == 8 ? 2 : 1))) void k_start(
    double* __restrict__ q, Grid g, LimParams lp, CflEos eos, double dn_min, double cflm, double* __restrict__ partial,
    double* __restrict__ dt_out, double* __restrict__ t_io) {
    __shared__ double red[4];
    __shared__ double last;
    double vmag = 0.;
    for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < g.N; c += (long)gridDim.x * blockDim.x) {
        double m[5][NB], v0;
#pragma unroll
        for (int r = 0; r < NB; r++)
#pragma unroll
            for (int f = 0; f < 5; f++) m[f][r] = q[((long)r * g.nQ + f) * g.N + c];
        const double cs = cell_sound_speed(q, g, c, eos, &v0);
        if (v0 > vmag && m[RH][0] > dn_min) vmag = v0;
        if (c == g.N - 1) {
            if (gridDim.x == 1) last = cs;
            else partial[gridDim.x] = cs;
        }
        if (limit_cell<NB, QP, 5>(m, lp)) {
#pragma unroll
            for (int r = 0; r < NB; r++)
#pragma unroll
                for (int f = 0; f < 5; f++) q[((long)r * g.nQ + f) * g.N + c] = m[f][r];
        }
    }
    vmag = block_max(vmag, red);
    if (threadIdx.x == 0) {
        if (gridDim.x == 1) store_dt(vmag, last, g, cflm, dt_out, t_io);
        else partial[blockIdx.x] = vmag;
    }
}

template <int NB, int QP>
__global__ __launch_bounds__(256, (NB == 4 ? 4 : (NB == 8 ? 2 : 1))) void k_limit(double* __restrict__ q, Grid g, LimParams lp) {
    const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= g.N) return;
    double m[5][NB];
#pragma unroll
    for (int r = 0; r < NB; r++)
#pragma unroll
        for (int f = 0; f < 5; f++) m[f][r] = q[((long)r * g.nQ + f) * g.N + c];
    if (limit_cell<NB, QP, 5>(m, lp)) {
#pragma unroll
        for (int r = 0; r < NB; r++)
#pragma unroll
            for (int f = 0; f < 5; f++) q[((long)r * g.nQ + f) * g.N + c] = m[f][r];
    }
}

// ------------------------------------------------------------ kernel -------
__device__ __forceinline__ void fence() { asm volatile("" ::: "memory"); }

// A face's lift onto mode r in direction D is Lface(deg_D(r), side) times one
// face moment, sum_p w2_p b_k(p) F_p, k the mode's face-polynomial pair:
template <int NB, int D>
HD_DEV constexpr int lift_k(int r) {
    return pair_index(deg<NB>(r, row_axis(D)), deg<NB>(r, col_axis(D)));
}
}  // namespace fz


// The 13-moment cell kernel of the table-driven path: the face arrays hold the
// point fluxes of k_face_flux.
template <int NB, int QP>
__global__ __launch_bounds__(CELL13_WAVES * 64) void k_cell13(
    const double* __restrict__ qin, const double* __restrict__ qn, double* __restrict__ qout,
    const double* __restrict__ flx, const double* __restrict__ fly, const double* __restrict__ flz,
    const Tables* __restrict__ T, Grid g, Phys ph, StageParams sp) {
    constexpr int NQ = 13, NF = QP * QP, NPG = QP * QP * QP;
    constexpr int NS = (NB > 4) ? 12 : 3;
    constexpr int NCH = NF;  // volume points per exchange: one plane of the 3D rule
    static_assert(NCH <= CELL13_WAVES, "one wave per point computes the primitives");
    __shared__ double qp_s[NQ][NCH][64];
    __shared__ double pr_s[NCH][NPRIM13][64];
    const int f = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63);
    const long c = (long)xcd_block() * 64 + lane;  // XCD-contiguous ranges of cells
    const bool live = c < g.N;
    const long cc = live ? c : g.N - 1;  // lanes past the grid compute a copy of the last cell and store nothing
    // 32-bit position arithmetic: hd_create bounds the cells by 2^31
    const unsigned ucc = (unsigned)cc, cq = ucc / (unsigned)g.nx;
    const int i = (int)(ucc - cq * (unsigned)g.nx), j = (int)(cq % (unsigned)g.ny), k = (int)(cq / (unsigned)g.ny);
    double mf[NB];
#pragma unroll
    for (int r = 0; r < NB; r++) mf[r] = qin[qoff(g, cc, f, r)];
    const double dxi = g.dxi, dyi = g.dyi, dzi = g.dzi;
    // face lift of field f first, its loads beside those of the modes (one
    // memory phase instead of two), one direction at a time:
    // t[r] = dxi*sx[r] + dyi*sy[r] + dzi*sz[r] with the sums of k_cell
    const long fxm = (long)i + (long)(g.nx + 1) * ((long)j + (long)g.ny * k);
    const long fym = (long)i + (long)g.nx * ((long)j + (long)(g.ny + 1) * k);
    const long fzm = (long)i + (long)g.nx * ((long)j + (long)g.ny * k);
    const long nfx = (long)(g.nx + 1) * g.ny * g.nz, nfy = (long)g.nx * (g.ny + 1) * g.nz,
               nfz = (long)g.nx * g.ny * (g.nz + 1);
    double t[NB];
    lift13_dir<NB, NF, 0>(flx, nfx, fxm, fxm + 1, dxi, f, T, t);
    lift13_dir<NB, NF, 1>(fly, nfy, fym, fym + g.nx, dyi, f, T, t);
    lift13_dir<NB, NF, 2>(flz, nfz, fzm, fzm + (long)g.nx * g.ny, dzi, f, T, t);
    // ---- volume integral: every wave reaches every barrier ----
    // glf[r] = 0.25 cb[r] (t[r] - sum_d di acc_d[r]) for r >= 1, so each
    // accumulator starts at -t[r] over its grid factor and t[1..] need not
    // stay live through the volume loop (the kernel runs at 128 VGPRs)
    double acc[NS];
    {
        const double dx = 1. / dxi, dy = 1. / dyi, dz = 1. / dzi;
        acc[0] = -dx * t[KX];
        acc[1] = -dy * t[KY];
        acc[2] = -dz * t[KZ];
        if constexpr (NB > 4) {
            acc[3] = -dy * t[KYZ];
            acc[4] = 0.;
            acc[5] = -dx * t[KZX];
            acc[6] = 0.;
            acc[7] = -dx * t[KXY];
            acc[8] = 0.;
            if constexpr (NB == 10) {
                acc[9] = -dx * t[KXX];
                acc[10] = -dy * t[KYY];
                acc[11] = -dz * t[KZZ];
            } else {
                acc[9] = -dx * t[KXYZ];
                acc[10] = 0.;
                acc[11] = 0.;
            }
        }
    }
    const double t0 = t[0];
    // volume integral, NCH points per exchange: each wave writes its field's
    // point values, then reads the 13 values of each point; every wave
    // reaches every barrier
#pragma unroll 1
    for (int p0 = 0; p0 < NPG; p0 += NCH) {
#pragma unroll
        for (int q = 0; q < NCH; q++) {
            const double* b = T->bint[p0 + q];
            double v = 0.;
#pragma unroll
            for (int r = 0; r < NB; r++) v += b[r] * mf[r];
            qp_s[f][q][lane] = v;
        }
        __syncthreads();
        // the primitives of point f of the plane, once per point
        if (f < NCH) {
            double Qp[NQ], pr[NPRIM13];
#pragma unroll
            for (int e = 0; e < NQ; e++) Qp[e] = qp_s[e][f][lane];
            prim13(ph, Qp, pr);
#pragma unroll
            for (int e = 0; e < NPRIM13; e++) pr_s[f][e][lane] = pr[e];
        }
        __syncthreads();
#pragma unroll 1
        for (int q = 0; q < NCH; q++) {
            const int p = p0 + q;
            const double* b = T->bint[p];
            double Fx, Fy, Fz;
            flux13_field<NCH * 64>(ph, &qp_s[0][q][lane], &pr_s[q][0][lane], f, Fx, Fy, Fz);
            const double w = T->w3[p];
            acc[0] += w * Fx;
            acc[1] += w * Fy;
            acc[2] += w * Fz;
            if constexpr (NB > 4) {
                acc[3] += w * b[KZ] * Fy;
                acc[4] += w * b[KY] * Fz;
                acc[5] += w * b[KZ] * Fx;
                acc[6] += w * b[KX] * Fz;
                acc[7] += w * b[KY] * Fx;
                acc[8] += w * b[KX] * Fy;
                if constexpr (NB == 10) {
                    acc[9] += w * 3. * b[KX] * Fx;
                    acc[10] += w * 3. * b[KY] * Fy;
                    acc[11] += w * 3. * b[KZ] * Fz;
                } else {
                    acc[9] += w * b[KYZ] * Fx;
                    acc[10] += w * b[KZX] * Fy;
                    acc[11] += w * b[KXY] * Fz;
                }
            }
        }
        __syncthreads();  // the next plane overwrites qp_s and pr_s
    }
    if (!live) return;  // no barrier below
    double intr[NB];
    intr[0] = 0.;
    intr[KX] = 0.25 * T->cb[KX] * dxi * acc[0];
    intr[KY] = 0.25 * T->cb[KY] * dyi * acc[1];
    intr[KZ] = 0.25 * T->cb[KZ] * dzi * acc[2];
    if constexpr (NB > 4) {
        intr[KYZ] = 0.25 * T->cb[KYZ] * (dyi * acc[3] + dzi * acc[4]);
        intr[KZX] = 0.25 * T->cb[KZX] * (dxi * acc[5] + dzi * acc[6]);
        intr[KXY] = 0.25 * T->cb[KXY] * (dxi * acc[7] + dyi * acc[8]);
        if constexpr (NB == 10) {
            intr[KXX] = 0.25 * T->cb[KXX] * (dxi * acc[9]);
            intr[KYY] = 0.25 * T->cb[KYY] * (dyi * acc[10]);
            intr[KZZ] = 0.25 * T->cb[KZZ] * (dzi * acc[11]);
        } else {
            intr[KXYZ] = 0.25 * T->cb[KXYZ] * (dxi * acc[9] + dyi * acc[10] + dzi * acc[11]);
        }
    }
    double glf[NB];
    glf[0] = 0.25 * t0;
#pragma unroll
    for (int r = 1; r < NB; r++) glf[r] = -intr[r];
    // ---- source: explicit relaxation (ivis 0), body force ----
    double src[NB];
#pragma unroll
    for (int r = 0; r < NB; r++) src[r] = 0.;
    const double rate = f >= T_QX ? sp.coll_q : sp.coll;
    if (sp.ivis == 0 && f >= T_PXX && rate != 0.) {
#pragma unroll 1
        for (int r = 0; r < NB; r++) {
            double s = 0.;
#pragma unroll 1
            for (int p = 0; p < NPG; p++) {
                double qv = 0.;
#pragma unroll
                for (int rr = 0; rr < NB; rr++) qv += T->bint[p][rr] * mf[rr];
                s += T->bwint[p][r] * (-rate * qv);
            }
            src[r] = 0.125 * T->cb[r] * s;
        }
    }
    if (f >= MX && f <= MZ && sp.bf[f - MX] != 0.)
#pragma unroll
        for (int r = 0; r < NB; r++) src[r] += sp.bf[f - MX] * qin[qoff(g, c, RH, r)];
    if (f == EN && (sp.bf[0] != 0. || sp.bf[1] != 0. || sp.bf[2] != 0.))
#pragma unroll
        for (int r = 0; r < NB; r++)
            src[r] += sp.bf[0] * qin[qoff(g, c, MX, r)] + sp.bf[1] * qin[qoff(g, c, MY, r)] +
                      sp.bf[2] * qin[qoff(g, c, MZ, r)];
    // ---- update, SSP combination, NaN check of mode 1 ----
    if (sp.mode == 1) {
#pragma unroll
        for (int r = 0; r < NB; r++) qout[qoff(g, c, f, r)] = -(glf[r] - src[r]);
        return;
    }
    const double dt = *sp.dt;
    const double fac = f >= T_QX ? 1. / (1. + dt * sp.coll_q) : 1. / (1. + dt * sp.coll);
    bool bad = false;
#pragma unroll
    for (int r = 0; r < NB; r++) {
        double v = mf[r] - dt * (glf[r] - src[r]);
        if (sp.ivis == 1 && f >= T_PXX) v = fac * v;
        const long o = qoff(g, c, f, r);
        if (r == 0 && v != v) bad = true;
        if (sp.combine == 1) v = 0.5 * (qn[o] + v);
        else if (sp.combine == 2) v = 0.75 * qn[o] + 0.25 * v;
        else if (sp.combine == 3) v = (1. / 3.) * qn[o] + (2. / 3.) * v;
        qout[o] = v;
    }
    if (bad) {
        atomicOr(sp.err, 1);
        atomicMin(sp.bad, (unsigned long long)c);
    }
}

}  // namespace hd
