// hd_stage.h -- one RK stage of the fused path: a workgroup of waves per run
// of cells, the stage's parts spread over the waves.
//
// The operator is that of hd_fused.h (volume integral, Riemann fluxes on six
// faces, lifts, sources, update, SSP combination, the next stage's limiter).
// A tile is 64 consecutive positions of a plane's row lattice (nx+1 positions
// per row: the faces across x), one per lane; it updates the cells of its
// first 63 positions, so that the face above a cell in x is always the next
// lane's (thin grids: Rows below).  A workgroup steps its tile through planes of z:
//   part 0: the face below every cell in y, and the first third (half, with
//           two Gauss points) of the volume integral;
//   part 1: the face above in y, and the second third (half);
//   part 2: the faces in x, and the rest of the volume integral (with two
//           points: none);
//   part 3: the face above in z (the one below is the last plane's), then the
//           sum of all parts, the time step, the limiter and the stores.
// Every face is evaluated once, but for the faces in y (by the tiles on both
// sides) and the first one of a workgroup in z.  The parts meet once per plane;
// part 3 lets go of the others' sums before it takes the time step.
// Part 3 alone holds terms of the state: with the state in one of the partial
// sums each later addition rounded it once more (a step's error 1.3e-16 of the
// state against 0.4e-16 to 0.8e-16), for 0 to 10 % less time (vortex 1363 us a
// step against 1438, linear 3950 and 4040, 13 moments 6935 and 7080, channel
// 23.2 and 25.7).  Which wave takes which part rotates with the
// workgroup, so that what inequality there is does not always meet one SIMD.
//
// Fields of a face: the stress fields' flux is linear in the velocity, and a
// face of direction d carries only row d of the stress.  With stress a face
// therefore has eight values (rh..en and the row) and eight fluxes (rh..en
// and the velocity, from which the six stress rows follow), not eleven; with
// 13 moments also the heat flux along d and, for its flux, the temperature.
#pragma once
#include "hd_fused.h"

namespace hd {
namespace sg {

using fz::CellPos;

// values and moments of a face
HD_DEV constexpr int face_nm(int nq) { return nq == 13 ? 9 : (nq >= 11 ? 8 : 5); }
// Field of value e of a face of direction d: rh..en, the row of the stress,
// with 13 moments the heat flux along d.  The 13-moment pzz = -pxx - pyy has
// no field of its own (face_pzz): its value starts from pxx.
HD_DEV constexpr int face_field(int nq, int d, int e) {
    return e < 5 ? e
         : e == 8 ? T_QX + d
         : nq == 13 ? (d == 0 ? (e == 5 ? T_PXX : (e == 6 ? T_PXY : T_PXZ))
                     : d == 1 ? (e == 5 ? T_PXY : (e == 6 ? T_PYY : T_PYZ))
                              : (e == 5 ? T_PXZ : (e == 6 ? T_PYZ : T_PXX)))
         : d == 0 ? (e == 5 ? PXX : (e == 6 ? PXY : PXZ))
         : d == 1 ? (e == 5 ? PXY : (e == 6 ? PYY : PYZ))
                  : (e == 5 ? PXZ : (e == 6 ? PYZ : PZZ));
}
HD_DEV constexpr bool face_pzz(int nq, int d, int e) { return nq == 13 && d == 2 && e == 7; }
// stress P_da at a point with fields Q
template <int NQ>
__device__ __forceinline__ double stress_value(const double* Q, int d, int a) {
    if (NQ == 13 && d == 2 && a == 2) return -(Q[T_PXX] + Q[T_PYY]);
    return Q[face_field(NQ, d, 5 + a)];
}
// stochastic stress component of row d, column a
HD_DEV constexpr int noise_comp(int d, int a) {
    return d == a ? d : (d + a == 1 ? 3 : (d + a == 2 ? 4 : 5));
}
// Scalars whose fluxes drive the fields past en: the velocity, with 13 moments
// also the temperature.
HD_DEV constexpr int nscal(int nq) { return nq == 13 ? 4 : (nq >= 11 ? 3 : 1); }
// Factor of field f's flux in direction d from scalar a: colvis (4/3, -2/3 or
// 1) times u_a for the stress, col_q T along d for the heat flux; 0 if none.
HD_DEV constexpr bool drives(int nq, int f, int a, int d) {
    if (nq == 13 && f >= T_QX) return a == 3 && f - T_QX == d;
    if (a > 2 || f < 5) return false;
    const int ndiag = nq == 13 ? 2 : 3;
    if (f < 5 + ndiag) return a == d;
    const int off = f - 5 - ndiag;  // xy, xz, yz
    return a != d && off == (a + d == 1 ? 0 : (a + d == 2 ? 1 : 2));
}
__device__ __forceinline__ double drive_factor(const Phys& ph, int nq, int f, int a) {
    if (a == 3) return ph.colq;
    if (f < 5 + (nq == 13 ? 2 : 3)) return f - 5 == a ? ph.c4d3cv : -ph.c2d3cv;
    return ph.colvis;
}

// Pointer to cell c of plane `plane`, stepped plane by plane.  The empty asm
// hides where it came from, so that the compiler neither keeps the addresses
// of every plane alive nor shares them between the parts of the kernel.
typedef const __attribute__((address_space(1))) double* gptr;
typedef __attribute__((address_space(1))) double* gptr_w;
__device__ __forceinline__ gptr plane_ptr(const double* q, long N, int plane, long c) {
    asm volatile("" : "+v"(c));
    return (gptr)(q + (long)plane * N + c);
}
template <typename P>
__device__ __forceinline__ void step(P& p, long st) {
    p += st;
    asm volatile("" : "+v"(p));
}
// end of a section: no load or computation moves across
__device__ __forceinline__ void section() {
    fz::fence();
    fz::point_barrier();
}

// Values that are complete here: the compiler may not move their last
// operations to where they are used (it would keep the operands alive
// instead, hundreds of registers).
template <int A, int B>
__device__ __forceinline__ void pin(double (&v)[A][B]) {
#pragma unroll
    for (int a = 0; a < A; a++)
#pragma unroll
        for (int b = 0; b < B; b++) asm volatile("" : "+v"(v[a][b]));
}

template <int B>
__device__ __forceinline__ void pin(double (&v)[B]) {
#pragma unroll
    for (int b = 0; b < B; b++) asm volatile("" : "+v"(v[b]));
}

// LDS of a workgroup: two partial sums of a cell's right-hand side, one face's moments
template <int NB, int NQ>
HD_DEV constexpr int lds_doubles() { return (2 * NB * NQ + face_nm(NQ) * fz::face_nk<NB>()) * 64; }
// k_stage_wide has a CU to itself: the cells' state and step start in its LDS
// too, where they fit.
template <int NB, int NQ>
HD_DEV constexpr bool wide_staged() { return (lds_doubles<NB, NQ>() + 2 * NB * NQ * 64) * 8 <= 160 * 1024 - 64; }
template <int NB, int NQ>
HD_DEV constexpr int wide_lds_doubles() { return lds_doubles<NB, NQ>() + (wide_staged<NB, NQ>() ? 2 * NB * NQ * 64 : 0); }

// ------------------------------------------------------------- faces -------
// The modes that a DIR face needs of cell c.
template <int NB, int NQ, int DIR>
__device__ __forceinline__ void load_side(const double* __restrict__ q, long N, long c, double (&m)[face_nm(NQ)][NB]) {
    constexpr int NM = face_nm(NQ);
    gptr p = plane_ptr(q, N, 0, c);
#pragma unroll
    for (int r = 0; r < NB; r++)
#pragma unroll
        for (int f = 0; f < NQ; f++) {
#pragma unroll
            for (int e = 0; e < NM; e++) {
                if (face_field(NQ, DIR, e) == f) m[e][r] = face_pzz(NQ, DIR, e) ? -*p : *p;
                else if (face_pzz(NQ, DIR, e) && f == T_PYY) m[e][r] -= *p;
            }
            step(p, N);
        }
}

// The face basis b_k at point (ii, jj), selected in scalar registers: a table
// in memory costs a wait on the scalar cache at every point.
template <int NB, int QP>
struct FacePoint {
    double b[fz::face_nk<NB>()], w;
    __device__ __forceinline__ FacePoint(int ii, int jj) {
        constexpr double s = fz::Rule<QP>::x(QP - 1);
        if constexpr (QP == 2) {
            b[1] = ii ? s : -s;
            b[2] = jj ? s : -s;
            if constexpr (NB == 8) b[3] = ii == jj ? s * s : -(s * s);
            w = 1.0;
        } else {
            constexpr double w0 = fz::Rule<3>::w(0), w1 = fz::Rule<3>::w(1);
            b[1] = ii == 1 ? 0.0 : (ii == 0 ? -s : s);
            b[2] = jj == 1 ? 0.0 : (jj == 0 ? -s : s);
            b[3] = (ii == 1 || jj == 1) ? 0.0 : (ii == jj ? s * s : -(s * s));
            b[4] = ii == 1 ? fz::Rule<3>::p2(1) : fz::Rule<3>::p2(0);
            b[5] = jj == 1 ? fz::Rule<3>::p2(1) : fz::Rule<3>::p2(0);
            w = (ii == 1) != (jj == 1) ? w0 * w1 : (ii == 1 ? w1 * w1 : w0 * w0);
        }
        b[0] = 1.0;
    }
};
// A face polynomial at a point.  The transposes evaluate theirs by these too
// (fz::face_poly holds the same b_k): explicit fma, so that both sides of a
// Riemann problem are bitwise the same there.
template <int NK>
__device__ __forceinline__ double eval_one(const double* K, const double* b) {
    double s = K[0];
#pragma unroll
    for (int k = 1; k < NK; k++) s = fma(K[k], b[k], s);
    return s;
}
template <int NM, int NK>
__device__ __forceinline__ void eval_point(const double (&K)[NM][NK], const double (&b)[NK], double* out) {
#pragma unroll
    for (int e = 0; e < NM; e++) out[e] = eval_one<NK>(K[e], b);
}

// Face-polynomial coefficients of a DIR face from a cell's modes: the modes
// odd along DIR enter with sign sgn (+1 above the cell, -1 below).  No product
// but sgn's, so that nothing here can be contracted in two ways.
template <int NB, int NM, int DIR, int NK>
__device__ __forceinline__ void signed_coeffs(const double (&m)[NM][NB], double sgn, double (&K)[NM][NK]) {
#pragma unroll
    for (int e = 0; e < NM; e++)
#pragma unroll
        for (int k = 0; k < NK; k++) {
            double s = 0., odd = 0.;
            bool has = false, hodd = false;
#pragma unroll
            for (int r = 0; r < NB; r++) {
                if (fz::lift_k<NB, DIR>(r) != k) continue;
                if (fz::deg<NB>(r, DIR) == 1) {
                    odd = m[e][r];
                    hodd = true;
                } else {
                    s = has ? s + m[e][r] : m[e][r];
                    has = true;
                }
            }
            K[e][k] = hodd ? fma(sgn, odd, s) : s;
        }
}

// The face of direction DIR between cells cL and cR: its NM*NK moments, times
// dxi_d, in M.  extL/extR: that side is outside the grid
// (boundary kind bc) and follows from the other side's trace.
template <int NB, int QP, int NQ, int RM, bool NZ, int DIR>
__device__ __forceinline__ void face_moments(const double* __restrict__ q, const Grid& g, long cL, long cR, bool extL,
                                             bool extR, int bc, const CellPos& cp, long fid, const Phys& ph,
                                             double dxi_d, const StageParams& sp,
                                             double (&M)[face_nm(NQ)][fz::face_nk<NB>()]) {
    constexpr int NF = QP * QP, NM = face_nm(NQ), NK = fz::face_nk<NB>();
    double KL[NM][NK], KR[NM][NK];
    {
        // both sides' loads before the first use
        double mL[NM][NB], mR[NM][NB];
        load_side<NB, NQ, DIR>(q, g.N, cL, mL);
        load_side<NB, NQ, DIR>(q, g.N, cR, mR);
        // a side outside the grid starts as a copy of the other side's trace
        signed_coeffs<NB, NM, DIR, NK>(mL, extL ? -1.0 : 1.0, KL);
        signed_coeffs<NB, NM, DIR, NK>(mR, extR ? 1.0 : -1.0, KR);
        pin(KL);
        pin(KR);
        section();
    }
    const bool ext = extL || extR;
    bool zero_normal = false;
    if (ext) {
        // outflow boundaries decide on the whole face (src/boundary.f90:213-338)
        if (bc == BC_OUTFLOW && !(DIR == 0 && extR)) {
            double v = 0.;
            for (int p = 0; p < NF; p++) {
                const FacePoint<NB, QP> fp(p / QP, p % QP);
                const double s = eval_one<NK>(KL[MX + DIR], fp.b);
                v = (p == 0) ? s : (extR ? fmin(v, s) : fmax(v, s));
            }
            zero_normal = extR ? (v < 0.0) : (v > 0.0);
        }
    }
#pragma unroll
    for (int e = 0; e < NM; e++)
#pragma unroll
        for (int k = 0; k < NK; k++) M[e][k] = 0.;
    // the row of the stochastic stress, one point ahead of its use
    float Sn[3];
    if constexpr (NZ) {
#pragma unroll
        for (int a = 0; a < 3; a++) Sn[a] = sp.noise[DIR][((long)a * NF) * sp.nfb + fid];
    }
    int ii = 0, jj = 0;
#pragma unroll 1
    for (int p = 0; p < NF; p++) {
        const FacePoint<NB, QP> fp(ii, jj);
        if (++jj == QP) {
            jj = 0;
            ii++;
        }
        double QL[NM], QR[NM], F[NM];
        eval_point<NM, NK>(KL, fp.b, QL);
        eval_point<NM, NK>(KR, fp.b, QR);
        if (ext) {
            if (bc == BC_NOSLIP) {
                if (extL) QL[MX] = QL[MY] = QL[MZ] = 0.0;
                else QR[MX] = QR[MY] = QR[MZ] = 0.0;
            } else if (bc == BC_WALL || (bc == BC_OUTFLOW && zero_normal)) {
                if (extL) QL[MX + DIR] = 0.0;
                else QR[MX + DIR] = 0.0;
            } else if (bc == BC_OUTFLOW && DIR == 0 && extR) {
                if (QR[MX] > 0.0) QR[MX] = -QL[MX];
            }
            if constexpr (DIR == 0) {
                // x_bc_inflow (src/boundary.f90:571-592): prescribed rh, mx, en;
                // no transverse momentum; the stress fields from the interior
                if (bc == BC_INFLOW && extL) fz::inflow_ghost<NQ>(sp.inflow, g, cp, p, NF, QL);
            }
        }
        double S[3] = {0., 0., 0.};
        if constexpr (NZ) {
            const int pn = p + 1 < NF ? p + 1 : p;
#pragma unroll
            for (int a = 0; a < 3; a++) {
                S[a] = Sn[a];
                Sn[a] = sp.noise[DIR][((long)a * NF + pn) * sp.nfb + fid];
            }
        }
        pr::face_flux<NQ, DIR, RM, NZ>(ph, QL, QR, S, F);
        const double wd = QP == 2 ? dxi_d : fp.w * dxi_d;
#pragma unroll
        for (int e = 0; e < NM; e++) {
            F[e] *= wd;
            M[e][0] += F[e];
#pragma unroll
            for (int k = 1; k < NK; k++) M[e][k] = fma(fp.b[k], F[e], M[e][k]);
        }
    }
    pin(M);
}
template <int NM, int NK>
__device__ __forceinline__ void store_moments(const double (&M)[NM][NK], double* __restrict__ mom) {
#pragma unroll
    for (int e = 0; e < NM; e++)
#pragma unroll
        for (int k = 0; k < NK; k++) mom[(e * NK + k) * 64] = M[e][k];
}

// ------------------------------------------------------------ volume -------
// Index of mode r among the modes with degree >= 1 along d
template <int NB>
HD_DEV constexpr int ndeg() { return NB == 4 ? 1 : 4; }
template <int NB>
HD_DEV constexpr int deg_index(int d, int r) {
    int n = 0;
    for (int s = 0; s < r; s++)
        if (fz::deg<NB>(s, d) > 0) n++;
    return n;
}

// A uniform value in scalar registers.
__device__ __forceinline__ double scalar(double x) {
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)b);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Fluxes at volume point (i,j,k) from the point's fields Q, projected onto
// the modes' derivatives; the products are written as fma so that the
// compiler does not share scaled modes between points (which would keep
// hundreds of them alive).  HYD: rh..en into rhs; VEL: the scalars into au.
template <int NB, int QP, int NQ, bool NZ, bool HYD, bool VEL>
__device__ __forceinline__ void volume_point(const double (&Q)[HYD ? NQ : (NQ == 13 ? 5 : 4)], int i, int j, int k, double (&rhs)[5][NB],
                                             double (&au)[nscal(NQ)][3][ndeg<NB>()], const Phys& ph,
                                             const double (&di)[3], const StageParams& sp, long c, long N) {
    float S[6];
    if constexpr (NZ && HYD) {
        constexpr long npg = QP * QP * QP;
#pragma unroll
        for (int e = 0; e < 6; e++) S[e] = sp.noise[3][((long)e * npg + (i * QP + j) * QP + k) * N + c];
    }
    const double ri = pr::rcp(Q[RH]);
    const double u[3] = {Q[MX] * ri, Q[MY] * ri, Q[MZ] * ri};
    double P = 0.;
    if constexpr (HYD || NQ == 13) {
        P = ph.gm1 * (Q[EN] - 0.5 * (Q[MX] * u[0] + Q[MY] * u[1] + Q[MZ] * u[2]));
        P = P < ph.P_floor ? ph.P_floor : P;
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double wd = QP == 2 ? di[d] : scalar(fz::Rule<QP>::w3(i, j, k) * di[d]);
        const double ud = wd * u[d];
        double F[5];
        if constexpr (HYD) {
            F[RH] = wd * Q[MX + d];
            F[EN] = (Q[EN] + P) * ud;
        }
        if constexpr (HYD && NQ >= 11) {
            double Pn[3];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                Pn[a] = stress_value<NQ>(Q, d, a);
                if constexpr (NZ) Pn[a] -= (double)S[noise_comp(d, a)];
                F[MX + a] = fma(Q[MX + a], ud, wd * (a == d ? Pn[a] + P : Pn[a]));
            }
            double pu = fma(Pn[0], u[0], fma(Pn[1], u[1], Pn[2] * u[2]));
            if constexpr (NQ == 13) pu += Q[T_QX + d];
            F[EN] = fma(wd, pu, F[EN]);
        } else if constexpr (HYD) {
#pragma unroll
            for (int a = 0; a < 3; a++) F[MX + a] = a == d ? fma(Q[MX + a], ud, wd * P) : Q[MX + a] * ud;
        }
        // dphi_r/dxi_d at the point: 1, other coordinates, or 3 x_d
#pragma unroll
        for (int r = 1; r < NB; r++) {
            if (fz::deg<NB>(r, d) == 0) continue;
            const double cf = fz::dphi<NB, QP>(d, r, i, j, k);
            if (cf == 0.0) continue;
            if constexpr (HYD) {
#pragma unroll
                for (int f = 0; f < 5; f++) rhs[f][r] = fma(cf, F[f], rhs[f][r]);
            }
            if constexpr (VEL) {
#pragma unroll
                for (int a = 0; a < 3; a++)
                    au[a][d][deg_index<NB>(d, r)] = fma(cf, a == d ? ud : wd * u[a], au[a][d][deg_index<NB>(d, r)]);
                if constexpr (NQ == 13)
                    au[3][d][deg_index<NB>(d, r)] = fma(cf, wd * (P * ri), au[3][d][deg_index<NB>(d, r)]);
            }
        }
    }
    fz::point_barrier();
}

// innerintegral2 (src/flux.f90:751-928) of cell c without its 0.25 cb_r; with
// stress, the fluxes of the fields past en are carried by their scalars'
// projections au[a][d][.] onto the modes that vary along d.  nbasis 10 holds one x plane
// of the cell at a time (its polynomial in y and z, six coefficients a
// field) and reads the modes once per plane, since modes and accumulators
// together do not fit 256 registers.  I0, I1: the x planes of the rule to take.
template <int NB, int QP, int NQ, bool NZ, bool HYD, bool VEL, int I0, int I1>
__device__ __forceinline__ void volume_moments(const double* __restrict__ q, const Grid& g, long c,
                                               double (&rhs)[5][NB], double (&au)[nscal(NQ)][3][ndeg<NB>()],
                                               const Phys& ph, const StageParams& sp) {
    const double di[3] = {g.dxi, g.dyi, g.dzi};
    constexpr int NV = HYD ? NQ : (NQ == 13 ? 5 : 4);  // fields read
    if constexpr (NB == 10) {
#pragma unroll
        for (int i = I0; i < I1; i++) {
            const double x = fz::Rule<QP>::x(i), p2 = fz::Rule<QP>::p2(i);
            double a0[NV], ay[NV], az[NV], ayz[NV], ayy[NV], azz[NV];
#pragma unroll
            for (int f = 0; f < NV; f++) {
                gptr p = plane_ptr(q, g.N, f, c);
                double m[NB];
#pragma unroll
                for (int r = 0; r < NB; r++) {
                    m[r] = *p;
                    step(p, (long)NQ * g.N);
                }
                a0[f] = fma(p2, m[KXX], m[0]);
                if (x != 0.0) a0[f] = fma(x, m[KX], a0[f]);
                ay[f] = x != 0.0 ? fma(x, m[KXY], m[KY]) : m[KY];
                az[f] = x != 0.0 ? fma(x, m[KZX], m[KZ]) : m[KZ];
                ayz[f] = m[KYZ];
                ayy[f] = m[KYY];
                azz[f] = m[KZZ];
                if (f % 3 == 2 || f == NV - 1) section();
            }
#pragma unroll
            for (int j = 0; j < QP; j++) {
                const double y = fz::Rule<QP>::x(j), q2 = fz::Rule<QP>::p2(j);
#pragma unroll
                for (int k = 0; k < QP; k++) {
                    const double z = fz::Rule<QP>::x(k), r2 = fz::Rule<QP>::p2(k);
                    double Q[NV];
#pragma unroll
                    for (int f = 0; f < NV; f++) {
                        double s = fma(q2, ayy[f], a0[f]);
                        if (y != 0.0) s = fma(y, ay[f], s);
                        s = fma(r2, azz[f], s);
                        if (z != 0.0) s = fma(z, az[f], s);
                        if (y * z != 0.0) s = fma(y * z, ayz[f], s);
                        Q[f] = s;
                    }
                    volume_point<NB, QP, NQ, NZ, HYD, VEL>(Q, i, j, k, rhs, au, ph, di, sp, c, g.N);
                }
            }
        }
    } else {
        double m[NQ][NB];
        fz::load_modes<NB, NQ>(q, g, c, m);
#pragma unroll
        for (int i = I0; i < I1; i++)
#pragma unroll
            for (int j = 0; j < QP; j++)
#pragma unroll
                for (int k = 0; k < QP; k++) {
                    double Q[NQ];
#pragma unroll
                    for (int f = 0; f < NQ; f++) {
                        double s = m[f][0];
#pragma unroll
                        for (int r = 1; r < NB; r++) s = fma(fz::phi_int<NB, QP>(r, i, j, k), m[f][r], s);
                        Q[f] = s;
                    }
                    volume_point<NB, QP, NQ, NZ, HYD, VEL>(Q, i, j, k, rhs, au, ph, di, sp, c, g.N);
                }
    }
}

// advance_time_level and the SSP combination (src/integrator.f90:62-86,
// 210-232) of a value m of the stage's input, its right-hand side and the
// step-start value q0: v = fac (m + dt rhs), out = wn q0 + wv v.  The sums of
// the right-hand side hold no term of the state, so that the state is rounded
// where the formula rounds it, and nowhere else: in v, in wn q0 and in the
// combination.
struct Weights {
    double dt, fac[3];  // of rh..en, stress, heat flux
    double wn, wv;
    bool rhs;           // the right-hand side alone
};
template <int NQ>
HD_DEV constexpr int field_class(int f) { return f < 5 ? 0 : (NQ == 13 && f >= T_QX ? 2 : 1); }
template <int NQ>
__device__ __forceinline__ Weights stage_weights(const StageParams& sp) {
    Weights w;
    w.rhs = sp.mode == 1;
    w.wv = sp.combine == 0 ? 1. : (sp.combine == 1 ? 0.5 : (sp.combine == 2 ? 0.25 : 2. / 3.));
    w.wn = sp.combine == 0 ? 0. : (sp.combine == 1 ? 0.5 : (sp.combine == 2 ? 0.75 : 1. / 3.));
    w.dt = 0.;
    w.fac[0] = w.fac[1] = w.fac[2] = 1.;
    if (w.rhs) return w;
    const double* pdt = sp.dt;
    asm volatile("" : "+s"(pdt));  // read where it is used, not kept in registers across the planes
    w.dt = *pdt;
    if constexpr (NQ >= 11) {
        if (sp.ivis == 1) {
            w.fac[1] = 1. / (1. + w.dt * sp.coll);
            if constexpr (NQ == 13) w.fac[2] = 1. / (1. + w.dt * sp.coll_q);
        }
    }
    return w;
}
template <int NB, int NQ>
__device__ __forceinline__ void load_field(const double* __restrict__ q, const Grid& g, long c, int f, double (&m)[NB]) {
    gptr p = plane_ptr(q, g.N, f, c);
#pragma unroll
    for (int r = 0; r < NB; r++) {
        m[r] = *p;
        step(p, (long)NQ * g.N);
    }
}
// The right-hand side t of field f becomes its output: sources, time step,
// combination with the step-start values q0.
template <int NB, int NQ>
__device__ __forceinline__ void advance_field(const double* __restrict__ qin, const Grid& g, const StageParams& sp,
                                              const Weights& w, long c, int f, const double (&m)[NB],
                                              const double (&q0)[NB], double (&t)[NB]) {
    const long st = (long)NQ * g.N;
    // sources (src/sources.f90:12-84): ivis 0 relaxes the stress explicitly
    // (-coll*P, projected exactly in modal space); body force rho*g, m.g
    if constexpr (NQ >= 11) {
        const double rate = field_class<NQ>(f) == 2 ? sp.coll_q : sp.coll;
        if (f >= 5 && sp.ivis == 0 && rate != 0.)
#pragma unroll
            for (int r = 0; r < NB; r++) t[r] = fma(-rate, m[r], t[r]);
    }
    if (f >= MX && f <= MZ && sp.bf[f - MX] != 0.) {
        gptr p = plane_ptr(qin, g.N, RH, c);
#pragma unroll
        for (int r = 0; r < NB; r++) {
            t[r] = fma(sp.bf[f - MX], *p, t[r]);
            step(p, st);
        }
    }
    if (f == EN && (sp.bf[0] != 0. || sp.bf[1] != 0. || sp.bf[2] != 0.)) {
        gptr p = plane_ptr(qin, g.N, MX, c);
#pragma unroll
        for (int r = 0; r < NB; r++) {
            t[r] = fma(sp.bf[0], p[0], fma(sp.bf[1], p[g.N], fma(sp.bf[2], p[2 * g.N], t[r])));
            step(p, st);
        }
    }
    if constexpr (NB == 10) {
        // selects: branches would cost registers (13 moments, 96^3 cells: 7050 us
        // a step against 7330)
        const double fac = w.fac[field_class<NQ>(f)];
#pragma unroll
        for (int r = 0; r < NB; r++) {
            double v = fma(w.dt, t[r], m[r]);
            if (f >= 5) v *= fac;
            t[r] = w.rhs ? t[r] : (w.wn != 0. ? fma(w.wv, v, w.wn * q0[r]) : v);
        }
    } else {
        // branches, which the empty asm keeps from becoming selects (channel of
        // 64x128 cells: 25.7 us a step against 26.5)
        if (w.rhs) return;
#pragma unroll
        for (int r = 0; r < NB; r++) t[r] = fma(w.dt, t[r], m[r]);
        if (f >= 5 && sp.ivis == 1) {
            asm volatile("");
#pragma unroll
            for (int r = 0; r < NB; r++) t[r] *= w.fac[field_class<NQ>(f)];
        }
        if (w.wn != 0.) {
            asm volatile("");
#pragma unroll
            for (int r = 0; r < NB; r++) t[r] = fma(w.wv, t[r], w.wn * q0[r]);
        }
    }
}

template <int NB, int NK, int D, bool LO>
__device__ __forceinline__ void lift(const double (&m)[NK], double (&t)[NB]) {
#pragma unroll
    for (int r = 0; r < NB; r++) {
        const double x = m[fz::lift_k<NB, D>(r)];
        t[r] += LO && fz::deg<NB>(r, D) != 1 ? x : -x;
    }
}
// Field f's share of a part, without 0.25 cb_r: t (rh..en) or, for the fields
// past en, what the scalars' lifts tu in direction D and their volume
// projections au (VOL) drive.
template <int NB, int NQ, int D, bool VOL>
__device__ __forceinline__ void part_field(const Phys& ph, const double (&t)[5][NB], const double (&tu)[nscal(NQ)][NB],
                                           const double (&au)[nscal(NQ)][3][ndeg<NB>()], int f, double (&o)[NB]) {
    if (f < 5) {
#pragma unroll
        for (int r = 0; r < NB; r++) o[r] = t[f][r];
        return;
    }
#pragma unroll
    for (int r = 0; r < NB; r++) o[r] = 0.;
    if constexpr (NQ >= 11) {
#pragma unroll
        for (int a = 0; a < nscal(NQ); a++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                if (!drives(NQ, f, a, d)) continue;
                const double cf = drive_factor(ph, NQ, f, a);
                if constexpr (VOL) {
#pragma unroll
                    for (int r = 0; r < NB; r++)
                        if (fz::deg<NB>(r, d) > 0) o[r] = fma(cf, au[a][d][deg_index<NB>(d, r)], o[r]);
                }
                if (d == D)
#pragma unroll
                    for (int r = 0; r < NB; r++) o[r] = fma(cf, tu[a][r], o[r]);
            }
    }
}

template <int NB, int NQ>
__device__ __forceinline__ void store_field(double* __restrict__ qout, const Grid& g, long c, int f,
                                            const double (&v)[NB]) {
    gptr_w p = (gptr_w)plane_ptr(qout, g.N, f, c);
#pragma unroll
    for (int r = 0; r < NB; r++) {
        *p = v[r];
        step(p, (long)NQ * g.N);
    }
}

// ------------------------------------------------------------- waves -------
// How the cells are cut into tiles.  A tile is cut from the rows of one plane
// and steps through planes, the same for all its lanes.  A grid that is thin
// across x and y would leave lanes idle (a column of cells along z 63 of 64): it
// is FOLDed.  The planes are then taken in segments of zc; the rows of all
// segments (row j of segment n is row j + ny n) make one list, cut into tiles
// whatever the segments, and a tile steps each lane through its own segment.
// Rows have nx+1 positions, the last a face alone; folded rows that are periodic
// and of up to eight cells are packed whole, without it: a row's last cell has
// its face above in the row's first lane.
// us a step of 65,536 cells, folded against cut from planes: 1x1x65536 cells
// nbasis 4 52 / 1446, nbasis 10 216 / 7228; 4x4x4096 51 / 130, 194 / 533.
// The lane's own plane costs registers: 256x256x128 cells nbasis 4 4.37 ms
// folded, 3.95 ms cut from planes.
struct Rows {
    unsigned pitch, n;  // positions of a row, of a tile
    bool whole;
};
template <bool FOLD>
__host__ __device__ __forceinline__ Rows tile_rows(const Grid& g) {
    Rows o;
    o.whole = FOLD && g.nx <= 8 && g.bc[0] == BC_PERIODIC;
    o.pitch = (unsigned)g.nx + (o.whole ? 0u : 1u);
    o.n = o.whole ? 64u - 64u % (unsigned)g.nx : 63u;
    return o;
}
// tiles of nrow rows: the last position has no cell where rows have an extra one
template <bool FOLD>
inline long row_tiles(const Grid& g, long nrow) {
    const Rows o = tile_rows<FOLD>(g);
    return (o.pitch * nrow - (o.whole ? 0 : 1) + o.n - 1) / o.n;
}
inline long plane_tiles(const Grid& g) { return row_tiles<false>(g, g.ny); }
inline long fold_tiles(const Grid& g, int zc) { return row_tiles<true>(g, (long)g.ny * ((g.nz + zc - 1) / zc)); }
// planes that a folded tile steps through: fewer than zc if all of its cells are
// in the last segment
__device__ __forceinline__ int fold_planes(const Grid& g, unsigned tile, int zc) {
    const Rows o = tile_rows<true>(g);
    const int k0 = (int)(tile * o.n / o.pitch / (unsigned)g.ny) * zc;
    return g.nz - k0 < zc ? g.nz - k0 : zc;
}

// A lane's column of cells: position pi of its row at row j, planes stepped by
// the caller: k, or folded the segment's k0 + 0, 1, ..
struct Column {
    int pi, i, j;     // position 0..nx (the face below cell pi in x), cell, row
    int k0, next;     // folded: first plane; the lane that has the face above in x
    bool live;        // the lane updates the cell
    long row0;        // offset of the row within a plane
};
template <bool FOLD>
__device__ __forceinline__ Column column(const Grid& g, unsigned tile, int zc, int lane) {
    // 32-bit position arithmetic: 2^31 cells would not fit the device.
    // Worked out where it is used: kept across the planes it would cost registers
    // that the faces need.
    asm volatile("" : "+s"(tile));
    const Rows t = tile_rows<FOLD>(g);
    Column o;
    unsigned pos = tile * t.n + (unsigned)lane, row;
    if constexpr (FOLD) {
        const unsigned nrow = (unsigned)g.ny * (unsigned)((g.nz + zc - 1) / zc);
        if (t.whole && (unsigned)lane >= t.n) pos = tile * t.n;
        row = pos / t.pitch;
        o.pi = (int)(pos - row * t.pitch);
        o.live = row < nrow && o.pi < g.nx && (unsigned)lane < t.n;
        if (row >= nrow) row = nrow - 1u;
        const unsigned n = row / (unsigned)g.ny;
        row -= n * (unsigned)g.ny;
        o.k0 = (int)n * zc;
        o.next = t.whole && o.pi == g.nx - 1 ? lane - o.pi : (lane + 1) & 63;
    } else {
        const unsigned npos = t.pitch * (unsigned)g.ny;
        const bool in = pos < npos;
        if (!in) pos = npos - 1u;
        row = pos / t.pitch;
        o.pi = (int)(pos - row * t.pitch);
        o.live = in && o.pi < g.nx && lane < 63;
        o.k0 = 0;
        o.next = (lane + 1) & 63;
    }
    o.i = o.pi < g.nx ? o.pi : g.nx - 1;
    o.j = (int)row;
    o.row0 = (long)g.nx * o.j;
    return o;
}
// its plane kk, folded the last one past the grid's end
template <bool FOLD>
__device__ __forceinline__ int column_plane(const Grid& g, const Column& o, int kk) {
    if constexpr (!FOLD) return kk;
    return o.k0 + kk < g.nz ? o.k0 + kk : g.nz - 1;
}

// Face s (0 below, 1 above) in direction DIR of the column's cell at plane k
// (DIR 0: the face below lattice position pi, s = 0).
template <int NB, int QP, int NQ, int RM, bool NZ, int DIR>
__device__ __forceinline__ void column_face(const double* __restrict__ qin, const Grid& g, const Phys& ph,
                                            const StageParams& sp, const Column& o, int k, int s,
                                            double (&M)[face_nm(NQ)][fz::face_nk<NB>()]) {
    const long plane = (long)g.nx * g.ny;
    const int n = DIR == 0 ? g.nx : DIR == 1 ? g.ny : g.nz;
    const int af = DIR == 0 ? o.pi : (DIR == 1 ? o.j : k) + s;  // the face below cell af
    const bool per = g.bc[2 * DIR] == BC_PERIODIC;
    const bool extL = !per && af == 0, extR = !per && af == n;
    const int aL = af == 0 ? (per ? n - 1 : 0) : af - 1, aR = af == n ? (per ? 0 : n - 1) : af;
    const int bc = extL ? g.bc[2 * DIR] : g.bc[2 * DIR + 1];
    long base, st;
    if (DIR == 0) base = o.row0 + plane * k, st = 1;
    else if (DIR == 1) base = o.i + plane * k, st = g.nx;
    else base = o.row0 + o.i, st = plane;
    const long nfx = g.nx + 1, nfxy = nfx * (g.ny + 1);
    const int an = per && af == n ? 0 : af;
    const long fid = (DIR == 0 ? an : o.i) + nfx * (DIR == 1 ? an : o.j) + nfxy * (DIR == 2 ? an : k);
    CellPos cp;
    cp.i = o.i;
    cp.j = o.j;
    cp.k = k;
    cp.c = 0;
    face_moments<NB, QP, NQ, RM, NZ, DIR>(qin, g, base + aL * st, base + aR * st, extL, extR, bc, cp, fid, ph,
                                          DIR == 0 ? g.dxi : DIR == 1 ? g.dyi : g.dzi, sp, M);
}

// Waves per SIMD that the registers are held to.  With more modes than four and
// stress the sums' LDS leaves room for one workgroup a CU (nbasis 8, 11 fields,
// 64x64x48 cells: 855 us a step held to two, 760 to one).
HD_DEV constexpr int occupancy(int nb, int nq) { return nb == 4 && nq == 5 ? 3 : (nb > 4 && nq >= 11 ? 1 : 2); }
template <int NB, int NQ>
HD_DEV constexpr int occupancy() { return occupancy(NB, NQ); }

// Cost of items of zc planes on `resident` workgroups, in planes: rounds times
// an item's length, its start (the first face below in z and the first loads)
// worth 0.6 planes.
inline double march_cost(long items, int zc, long resident) {
    return (double)((items + resident - 1) / resident) * (zc + 0.6);
}

// A grid is folded if a quarter of the lanes would be idle otherwise.
inline bool stage_folds(const Grid& g) { return 3 * plane_tiles(g) * g.nz >= 4 * fold_tiles(g, 1); }

// How a grid is run: -1 by k_stage_wide, 0 in equal runs, n > 0 in items of n
// planes.
//  * Folded grids: the items of least cost; single planes where a plane is less
//    than a 128-byte line of cells, so that neighbouring lanes' cells follow each
//    other in memory (13 moments, 1x1x65536 cells: 650 us a step against 986 in
//    items of 4).
//  * Up to two tiles per CU k_stage_wide: latency decides (Sod tube of 256
//    cells 23.4 us a step in five waves against 24.7, channel 64x128 25.7
//    against 29.1).
//  * Up to 8 planes per resident workgroup in equal runs: whole rounds of items
//    would leave part of the chip idle (nbasis 10, 75x61x27: 350 us a step
//    against 461 in items of 4).
//  * Above, the items of least cost: neighbouring tiles at the same plane share
//    L2, which equal runs lose (nbasis 4, 256x256x128: 4.1 ms a step in items
//    of 8 or 16 against 5.0; nbasis 8, 120x80x64: 593 us in items of 8 against
//    637).
template <int NB, int NQ>
inline int stage_planes(const Grid& g, long cus) {
    const bool fold = stage_folds(g);
    const long tiles = plane_tiles(g), work = tiles * g.nz, resident = cus * occupancy<NB, NQ>();
    if (!fold && work <= 2 * cus && !(NB == 10 && NQ >= 11)) return -1;
    if (!fold && work < 8 * resident) return 0;
    if (fold && (long)g.nx * g.ny < 16) return 1;
    auto cost = [&](int zc) {
        return march_cost(fold ? fold_tiles(g, zc) : tiles * ((g.nz + zc - 1) / zc), zc, resident);
    };
    int best = 1;
    for (int zc = 2; zc <= g.nz && zc <= 16; zc++)
        if (cost(zc) < cost(best)) best = zc;
    return best;
}

// What the waves of a workgroup share.
struct Shared {
    double *r0, *r1;  // partial sums of the right-hand sides: parts 2 and 0, part 1
    double* z;        // moments of the face below in z
    double* m;        // k_stage_wide: the cells' state and step start
    int* flags;       // planes whose sums part 3 has read; planes that part 2 has written
};
__device__ __forceinline__ void raise(int* flag, int n) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __hip_atomic_store(flag, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// The waves of a workgroup are resident together, and the one waited for
// never waits for this one before it raises the flag.
__device__ __forceinline__ void await(int* flag, int n) {
    while (__hip_atomic_load(flag, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < n) __builtin_amdgcn_s_sleep(1);
}

// value of the next lane
__device__ __forceinline__ double next_lane(double x, int addr) {
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)b);
    const unsigned hi = (unsigned)__builtin_amdgcn_ds_bpermute(addr, (int)(unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Parts 0-2 of the tile's plane kk (p planes after the workgroup's first): one direction's
// face and a share of the volume integral; the sum to LDS.
template <int NB, int QP, int NQ, int RM, bool NZ, bool FOLD, int PART>
__device__ __forceinline__ void sum_part(const double* __restrict__ qin, const Grid& g, const Phys& ph,
                                         const StageParams& sp, unsigned tile, int zc, int kk, int p, const Shared& sh,
                                         int lane) {
    constexpr int NM = face_nm(NQ), NK = fz::face_nk<NB>();
    constexpr int D = PART == 2 ? 0 : 1;
    constexpr bool VOL = PART < QP;
    const Column o = column<FOLD>(g, tile, zc, lane);
    const int k = column_plane<FOLD>(g, o, kk);
    const long c = o.row0 + o.i + (long)g.nx * g.ny * k;
    double t[5][NB], tu[nscal(NQ)][NB], au[nscal(NQ)][3][ndeg<NB>()];
    {
        double M[NM][NK];
        column_face<NB, QP, NQ, RM, NZ, D>(qin, g, ph, sp, o, k, PART == 1 ? 1 : 0, M);
#pragma unroll
        for (int e = 0; e < NM; e++) {
            double s[NB];
#pragma unroll
            for (int r = 0; r < NB; r++) s[r] = 0.;
            if constexpr (PART == 0) {
                lift<NB, NK, 1, true>(M[e], s);
            } else if constexpr (PART == 1) {
                lift<NB, NK, 1, false>(M[e], s);
            } else {
                double h[NK];
                const int addr = o.next * 4;
#pragma unroll
                for (int n = 0; n < NK; n++) h[n] = next_lane(M[e][n], addr);
                lift<NB, NK, 0, true>(M[e], s);
                lift<NB, NK, 0, false>(h, s);
            }
#pragma unroll
            for (int r = 0; r < NB; r++) {
                if (e < 5) t[e < 5 ? e : 0][r] = s[r];
                else tu[e < 5 ? 0 : e - 5][r] = s[r];
            }
        }
        pin(t);
        if constexpr (NQ >= 11) pin(tu);
        section();
    }
#pragma unroll
    for (int a = 0; a < nscal(NQ); a++)
#pragma unroll
        for (int d = 0; d < 3; d++)
#pragma unroll
            for (int r = 0; r < ndeg<NB>(); r++) au[a][d][r] = 0.;
    if constexpr (VOL) {
        if constexpr (NB == 10 && NQ >= 11) {
            // in two passes over the points: their accumulators do not fit together
            volume_moments<NB, QP, NQ, NZ, true, false, PART, PART + 1>(qin, g, c, t, au, ph, sp);
            pin(t);
            section();
            volume_moments<NB, QP, NQ, NZ, false, true, PART, PART + 1>(qin, g, c, t, au, ph, sp);
        } else {
            volume_moments<NB, QP, NQ, NZ, true, (NQ >= 11), PART, PART + 1>(qin, g, c, t, au, ph, sp);
        }
        pin(t);
        if constexpr (NQ >= 11) {
#pragma unroll
            for (int a = 0; a < nscal(NQ); a++) pin(au[a]);
        }
        section();
    }
    double* const R = (PART == 1 ? sh.r1 : sh.r0) + lane;
    // part 2 is done first: it writes, part 0 adds
    if (PART == 0) await(sh.flags + 1, p + 1);
    else await(sh.flags, p);
#pragma unroll
    for (int f = 0; f < NQ; f++) {
        double v[NB];
        part_field<NB, NQ, D, VOL>(ph, t, tu, au, f, v);
#pragma unroll
        for (int r = 0; r < NB; r++) {
            double* const x = R + (f * NB + r) * 64;
            v[r] *= 0.25 * fz::cbasis<NB>(r);
            *x = PART == 0 ? *x + v[r] : v[r];
        }
        if (f % 4 == 3) section();
    }
    section();
    if (PART == 2) raise(sh.flags + 1, p + 1);
}

// Part 3 of the tile's plane kk after its face above in z (moments M, the next plane's
// face below): once all parts have met, the sum, the time step, the next
// stage's limiter and the stores.
template <int NB, int QP, int NQ, bool FOLD, bool WIDE>
__device__ __forceinline__ void finish_part(const double* __restrict__ qin, const double* __restrict__ qn,
                                            double* __restrict__ qout, const Grid& g, const Phys& ph, const StageParams& sp,
                                            unsigned tile, int zc, int kk, int p, long cell0,
                                            const Shared& sh, int lane, bool same,
                                            double (&M)[face_nm(NQ)][fz::face_nk<NB>()]) {
    constexpr int NM = face_nm(NQ), NK = fz::face_nk<NB>();
    Column o = column<FOLD>(g, tile, zc, lane);
    if constexpr (FOLD) o.live = o.live && o.k0 + kk < g.nz;
    const Weights w = stage_weights<NQ>(sp);
    const long c = o.row0 + o.i + (long)g.nx * g.ny * column_plane<FOLD>(g, o, kk);
    // Values of the state and the step start are loaded AHEAD fields before they
    // are used, the first ones before the parts meet.
    constexpr bool STAGED = WIDE && wide_staged<NB, NQ>();
    constexpr int AHEAD = NB == 4 ? 3 : (NB == 8 ? (NQ == 5 ? 2 : 3) : 1), RING = AHEAD + 1;
    double m[RING][NB], q0[RING][NB];
    const bool comb = sp.combine != 0 && sp.mode != 1;
    const double* const q0p = comb ? qn : qin;
    // the fields past en first: the limiter leaves them alone, so each is stored
    // as it comes
    auto load = [&](int i) {
        if (i >= NQ) return;
        const int f = (i + 5) % NQ;
        if constexpr (STAGED) {
#pragma unroll
            for (int r = 0; r < NB; r++) {
                m[i % RING][r] = sh.m[(f * NB + r) * 64 + lane];
                q0[i % RING][r] = sh.m[((NQ + f) * NB + r) * 64 + lane];
            }
        } else {
            load_field<NB, NQ>(qin, g, c, f, m[i % RING]);
            load_field<NB, NQ>(q0p, g, c, f, q0[i % RING]);
        }
    };
    if constexpr (NB < 10 && !STAGED)
#pragma unroll
        for (int i = 0; i < AHEAD; i++) load(i);
    double v[NQ][NB];
    __syncthreads();
    double* const z = sh.z + lane;
    // same: the faces below and above are one (a periodic axis of one cell)
    double tu[nscal(NQ)][NB];
#pragma unroll
    for (int e = 0; e < NM; e++) {
        double lo[NK], s[NB];
#pragma unroll
        for (int n = 0; n < NK; n++) {
            lo[n] = z[(e * NK + n) * 64];
            if (same) M[e][n] = lo[n];
        }
#pragma unroll
        for (int r = 0; r < NB; r++) s[r] = 0.;
        lift<NB, NK, 2, true>(lo, s);
        lift<NB, NK, 2, false>(M[e], s);
#pragma unroll
        for (int n = 0; n < NK; n++) z[(e * NK + n) * 64] = M[e][n];
#pragma unroll
        for (int r = 0; r < NB; r++) {
            if (e < 5) v[e < 5 ? e : 0][r] = (0.25 * fz::cbasis<NB>(r)) * s[r];
            else tu[e < 5 ? 0 : e - 5][r] = s[r];
        }
        if (NB > 4 && e % 2 == 1) section();
    }
    pin(tu);
#pragma unroll
    for (int f = 0; f < 5; f++) pin(v[f]);
    if constexpr (NB == 10 || STAGED)
#pragma unroll
        for (int i = 0; i < AHEAD; i++) load(i);
#pragma unroll
    for (int f = 0; f < NQ; f++) {
        if (f >= 5) {
#pragma unroll
            for (int r = 0; r < NB; r++) v[f][r] = 0.;
        }
        if constexpr (NQ >= 11) {
#pragma unroll
            for (int a = 0; a < nscal(NQ); a++) {
                if (!drives(NQ, f, a, 2)) continue;
                const double cf = drive_factor(ph, NQ, f, a);
#pragma unroll
                for (int r = 0; r < NB; r++) v[f][r] = fma(cf * (0.25 * fz::cbasis<NB>(r)), tu[a][r], v[f][r]);
            }
        }
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const int x = (f * NB + r) * 64 + lane;
            v[f][r] += sh.r0[x] + sh.r1[x];
        }
        if (!WIDE && f % (NB > 4 ? 2 : 4) == 1) section();
    }
    pin(v);
    raise(sh.flags, p + 1);
    section();
    bool bad = false;
#pragma unroll
    for (int i = 0; i < NQ; i++) {
        const int f = (i + 5) % NQ;
        load(i + AHEAD);
        advance_field<NB, NQ>(qin, g, sp, w, c, f, m[i % RING], q0[i % RING], v[f]);
        pin(v[f]);
        bad |= v[f][0] != v[f][0];
        if (NB > 4 && f >= 5 && o.live) store_field<NB, NQ>(qout, g, c, f, v[f]);
        if (!WIDE) section();
    }
    // When this output is the next stage's input, apply that stage's limiter
    // here: the reference limits the stage input in place before anything
    // reads it (src/integrator.f90:106-113), so the stored values are the same.
    if (sp.limit_out) fz::limit_cell<NB, QP, NQ>(v, sp.lp);
    if (!o.live) return;
#pragma unroll
    for (int f = 0; f < (NB > 4 ? 5 : NQ); f++) store_field<NB, NQ>(qout, g, c, f, v[f]);
    if (bad && !w.rhs) {
        atomicOr(sp.err, 1);
        atomicMin(sp.bad, (unsigned long long)(cell0 + c));
    }
}

// One tile over planes [k0, k1) (folded: of its segments, of zc planes), after p0
// planes of this workgroup: four waves.
template <int NB, int QP, int NQ, int RM, bool NZ, bool FOLD>
__device__ __forceinline__ void stage_march(const double* __restrict__ qin, const double* __restrict__ qn,
                                            double* __restrict__ qout, const Grid& g, const Phys& ph,
                                            const StageParams& sp, unsigned tile, int zc, int k0, int k1, int p0, int part,
                                            long cell0, const Shared& sh) {
    constexpr int NM = face_nm(NQ), NK = fz::face_nk<NB>();
    const int lane = (int)(threadIdx.x & 63u);
    if (part == 0) {
#pragma unroll 1
        for (int k = k0; k < k1; k++) {
            sum_part<NB, QP, NQ, RM, NZ, FOLD, 0>(qin, g, ph, sp, tile, zc, k, p0 + k - k0, sh, lane);
            __syncthreads();
        }
    } else if (part == 1) {
#pragma unroll 1
        for (int k = k0; k < k1; k++) {
            sum_part<NB, QP, NQ, RM, NZ, FOLD, 1>(qin, g, ph, sp, tile, zc, k, p0 + k - k0, sh, lane);
            __syncthreads();
        }
    } else if (part == 2) {
#pragma unroll 1
        for (int k = k0; k < k1; k++) {
            sum_part<NB, QP, NQ, RM, NZ, FOLD, 2>(qin, g, ph, sp, tile, zc, k, p0 + k - k0, sh, lane);
            __syncthreads();
        }
    } else {
        const bool one_z = g.nz == 1 && g.bc[4] == BC_PERIODIC;
#pragma unroll 1
        for (int k = k0; k <= k1; k++) {  // the face below plane k
            double M[NM][NK];
            if (k > k0 && one_z) {
#pragma unroll
                for (int e = 0; e < NM; e++)
#pragma unroll
                    for (int n = 0; n < NK; n++) M[e][n] = 0.;
            } else {
                const Column o = column<FOLD>(g, tile, zc, lane);
                const int kf = !FOLD ? k : (o.k0 + k < g.nz ? o.k0 + k : g.nz);
                column_face<NB, QP, NQ, RM, NZ, 2>(qin, g, ph, sp, o, kf, 0, M);
            }
            if (k == k0) {
#pragma unroll
                for (int e = 0; e < NM; e++)
#pragma unroll
                    for (int n = 0; n < NK; n++) sh.z[(e * NK + n) * 64 + lane] = M[e][n];
            } else {
                finish_part<NB, QP, NQ, FOLD, false>(qin, qn, qout, g, ph, sp, tile, zc, k - 1, p0 + k - 1 - k0, cell0, sh, lane,
                                               one_z, M);
            }
        }
    }
}

// k_stage_wide: a plane's state and step start to LDS for part 3, by the part
// that has least to do: part 2 with two points (no volume), else part 4.
template <int NB, int NQ>
__device__ __forceinline__ void bring_state(const double* __restrict__ qin, const double* __restrict__ qn,
                                            const Grid& g, const StageParams& sp, unsigned tile, int k,
                                            const Shared& sh, int lane) {
    const Column o = column<false>(g, tile, 1, lane);
    const long c = o.row0 + o.i + (long)g.nx * g.ny * k;
    double m[NQ][NB];
#pragma unroll
    for (int f = 0; f < NQ; f++) load_field<NB, NQ>(qin, g, c, f, m[f]);
    if (sp.combine != 0 && sp.mode != 1) {
        double q0[NQ][NB];
#pragma unroll
        for (int f = 0; f < NQ; f++) load_field<NB, NQ>(qn, g, c, f, q0[f]);
#pragma unroll
        for (int f = 0; f < NQ; f++)
#pragma unroll
            for (int r = 0; r < NB; r++) sh.m[((NQ + f) * NB + r) * 64 + lane] = q0[f][r];
    }
#pragma unroll
    for (int f = 0; f < NQ; f++)
#pragma unroll
        for (int r = 0; r < NB; r++) sh.m[(f * NB + r) * 64 + lane] = m[f][r];
}

// One tile of one plane by five waves, for grids of few tiles (latency): the
// face below in z has a wave of its own.
template <int NB, int QP, int NQ, int RM, bool NZ>
__device__ __forceinline__ void stage_wide(const double* __restrict__ qin, const double* __restrict__ qn,
                                           double* __restrict__ qout, const Grid& g, const Phys& ph,
                                           const StageParams& sp, unsigned tile, int k, int part, long cell0,
                                           const Shared& sh) {
    constexpr int NM = face_nm(NQ), NK = fz::face_nk<NB>();
    const int lane = (int)(threadIdx.x & 63u);
    if (part == 0) {
        sum_part<NB, QP, NQ, RM, NZ, false, 0>(qin, g, ph, sp, tile, 1, k, 0, sh, lane);
    } else if (part == 1) {
        sum_part<NB, QP, NQ, RM, NZ, false, 1>(qin, g, ph, sp, tile, 1, k, 0, sh, lane);
    } else if (part == 2) {
        sum_part<NB, QP, NQ, RM, NZ, false, 2>(qin, g, ph, sp, tile, 1, k, 0, sh, lane);
        if constexpr (wide_staged<NB, NQ>() && QP == 2) bring_state<NB, NQ>(qin, qn, g, sp, tile, k, sh, lane);
    } else {
        const bool one_z = g.nz == 1 && g.bc[4] == BC_PERIODIC;
        double M[NM][NK];
        if (part == 4 || !one_z) {
            const Column o = column<false>(g, tile, 1, lane);
            column_face<NB, QP, NQ, RM, NZ, 2>(qin, g, ph, sp, o, k, part == 3 ? 1 : 0, M);
        }
        if (part == 3) {
            finish_part<NB, QP, NQ, false, true>(qin, qn, qout, g, ph, sp, tile, 1, k, 0, cell0, sh, lane, one_z, M);
            return;
        }
#pragma unroll
        for (int e = 0; e < NM; e++)
#pragma unroll
            for (int n = 0; n < NK; n++) sh.z[(e * NK + n) * 64 + lane] = M[e][n];
        if constexpr (wide_staged<NB, NQ>() && QP == 3) bring_state<NB, NQ>(qin, qn, g, sp, tile, k, sh, lane);
    }
    __syncthreads();
}

// The workgroup's LDS, flags cleared.
template <int NB, int NQ>
__device__ __forceinline__ Shared share(double* lds, int* flags) {
    Shared sh;
    sh.r0 = lds;
    sh.r1 = lds + NB * NQ * 64;
    sh.z = lds + 2 * NB * NQ * 64;
    sh.m = lds + lds_doubles<NB, NQ>();
    sh.flags = flags;
    if (threadIdx.x < 2) flags[threadIdx.x] = 0;
    __syncthreads();
    return sh;
}

// The grid's work is ntile tiles of nz planes.  With zc > 0 a workgroup takes
// zc planes of one tile, tiles first, so that neighbouring tiles are at the
// same planes at the same time and find each other's modes in L2 (folded: one of
// the ntile tiles of segments of zc planes).  With zc = 0 it takes an equal run
// of the whole work, z fastest, in a launch of as many workgroups as are
// resident: they start and end together.  Workgroup b runs on XCD b mod 8: each
// XCD takes a contiguous eighth (the grid is a multiple of 8).
template <int NB, int QP, int NQ, int RM, bool NZ, bool FOLD>
__global__ __launch_bounds__(256, (occupancy<NB, NQ>())) void k_stage(
    const double* __restrict__ qin, const double* __restrict__ qn, double* __restrict__ qout, Grid g, Phys ph,
    StageParams sp, unsigned ntile, int zc) {
    __shared__ double lds[lds_doubles<NB, NQ>()];
    __shared__ int flags[2];
    const unsigned b = blockIdx.x >> 3, w = (blockIdx.x & 7u) * (gridDim.x >> 3) + b;
    if constexpr (FOLD) {
        if (w >= ntile) return;
        const Shared sh = share<NB, NQ>(lds, flags);
        const int part = __builtin_amdgcn_readfirstlane((int)(((threadIdx.x >> 6) + b) & 3u));
        stage_march<NB, QP, NQ, RM, NZ, true>(qin, qn, qout, g, ph, sp, w, zc, 0, fold_planes(g, w, zc), 0, part, 0, sh);
        return;
    }
    unsigned tile, left;
    int k0, p = 0;
    if (zc > 0) {
        const unsigned ch = w / ntile;
        tile = w - ch * ntile;
        k0 = (int)ch * zc;
        if (k0 >= g.nz) return;
        left = (unsigned)(k0 + zc < g.nz ? zc : g.nz - k0);
    } else {
        const unsigned long long work = (unsigned long long)ntile * (unsigned)g.nz;
        const unsigned long long u = work * w / gridDim.x;
        left = (unsigned)(work * (w + 1) / gridDim.x - u);
        tile = (unsigned)(u / (unsigned)g.nz);
        k0 = (int)(u - (unsigned long long)tile * (unsigned)g.nz);
    }
    const Shared sh = share<NB, NQ>(lds, flags);
    const int part = __builtin_amdgcn_readfirstlane((int)(((threadIdx.x >> 6) + b) & 3u));
#pragma unroll 1
    while (left > 0) {
        const int n = (unsigned)(g.nz - k0) < left ? g.nz - k0 : (int)left;
        stage_march<NB, QP, NQ, RM, NZ, false>(qin, qn, qout, g, ph, sp, tile, 0, k0, k0 + n, p, part, 0, sh);
        left -= (unsigned)n;
        p += n;
        k0 = 0;
        tile++;
    }
}

template <int NB, int QP, int NQ, int RM, bool NZ>
__global__ __launch_bounds__(320) void k_stage_wide(
    const double* __restrict__ qin, const double* __restrict__ qn, double* __restrict__ qout, Grid g, Phys ph,
    StageParams sp, unsigned ntile, unsigned nwork) {
    __shared__ double lds[wide_lds_doubles<NB, NQ>()];
    __shared__ int flags[2];
    const unsigned t = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (t >= nwork) return;
    const Shared sh = share<NB, NQ>(lds, flags);
    const unsigned k = t / ntile;
    const int part = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    stage_wide<NB, QP, NQ, RM, NZ>(qin, qn, qout, g, ph, sp, t - k * ntile, (int)k, part, 0, sh);
}

}  // namespace sg
}  // namespace hd
