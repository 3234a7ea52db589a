// hd_adjoint.h -- hand-written reverse mode (vector-Jacobian products) of the
// RK stage, for gradients of a run with respect to its initial state and the
// relaxation rate.
//
// For a stage  out = a*Q^n + b*v,  v = F_ivis(m + dt*R(m)),  R = -glflux + source
// (src/integrator.f90:62-252; F_ivis scales the stress fields by
// 1/(1 + dt*coll) when ivis = 1), the kernel k_stage_vjp computes, for one
// cell c,
//     lam_in[c] = sum_k w_k acc_k[c] + L'(raw)^T ( lp[c] + dt * sum_j (dR_j/dm_c)^T lp[j] )
// with lp = F_ivis'^T (b*lam_out): the transpose of the stage map applied to
// the cotangent of its output.  (dR/dm)^T is gathered per cell: the cell's
// own volume term, and for each of its six faces the face flux's Jacobian
// with respect to this cell's trace, applied to the cotangent that the face
// flux receives from both cells that use it (volume: innerintegral2,
// src/flux.f90:751-928; faces: calc_flux_x/y/z and flux_hllc,
// src/flux.f90:197-647; lift: glflux, src/flux.f90:932-1022; sources:
// src/sources.f90:12-84).  L' is the limiter (src/flux.f90:1077-1164) with
// its active set and factors frozen at the forward values: the factors that
// scaled the modes scale the cotangent.
//
// The point functions are differentiated by hand: the physical flux from
// primitives, Batten's HLLC with Davis speeds and the Roe solver
// (roe_point_vjp, hd_physics.h), each recomputing its forward intermediates and
// sweeping them backwards.  The traces (sg::signed_coeffs, sg::eval_point) and
// HLLC's speeds and branch (pr::side, pr::hllc_speeds) are the forward kernel's
// own functions: with stress HLLC's flux jumps where the contact speed changes
// sign, so the transpose must be of the branch that the forward stage took.
// The pressure floor and Roe's |eigenvalues| switch continuously and follow the
// transpose's own arithmetic (within rounding of the switch either one-sided
// derivative may be taken), as does Roe's test for a sound speed at all, which
// no state of positive pressure comes near.  The stochastic stress
// has no adjoint here.
#pragma once
#include "hd_stage.h"

namespace hd {
namespace adj {

// ---------------------------------------------------------------- flux ----
// reverse of flux_point13<DIR> (the 13-moment flux) from primitives:
// bF (cotangent of F) -> bQ (+=)
template <int DIR>
__device__ __forceinline__ void flux13_vjp(const Phys& ph, const double* Q, const pr::Prim& s, const double* bF,
                                           double* bQ) {
    constexpr int ND = MX + DIR;
    const double un = s.u[DIR];
    const double P = s.pf;
    // stress row DIR: indices of T_{DIR,a} (-1: t_zz = -t_xx - t_yy)
    const int trow[3][3] = {{T_PXX, T_PXY, T_PXZ}, {T_PXY, T_PYY, T_PYZ}, {T_PXZ, T_PYZ, -1}};
    double Tn[3];
#pragma unroll
    for (int a = 0; a < 3; a++) Tn[a] = trow[DIR][a] >= 0 ? Q[trow[DIR][a]] : -(Q[T_PXX] + Q[T_PYY]);
    double bun = bF[MX] * Q[MX] + bF[MY] * Q[MY] + bF[MZ] * Q[MZ] + bF[EN] * (Q[EN] + P);
    bun += (DIR == 0 ? ph.c4d3cv : -ph.c2d3cv) * bF[T_PXX] + (DIR == 1 ? ph.c4d3cv : -ph.c2d3cv) * bF[T_PYY];
    bQ[MX] += bF[MX] * un;
    bQ[MY] += bF[MY] * un;
    bQ[MZ] += bF[MZ] * un;
    bQ[EN] += bF[EN] * un;
    bQ[ND] += bF[RH];
    bQ[T_QX + DIR] += bF[EN];
    // heat-flux row: colq * P / rho
    const double bq = bF[T_QX + DIR] * ph.colq;
    const double bP = bF[ND] + bF[EN] * un + bq * s.ri;
    double bri = bq * P;
    double bu[3] = {bF[EN] * Tn[0], bF[EN] * Tn[1], bF[EN] * Tn[2]};
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double bt = bF[MX + a] + bF[EN] * s.u[a];
        if (trow[DIR][a] >= 0) {
            bQ[trow[DIR][a]] += bt;
        } else {
            bQ[T_PXX] -= bt;
            bQ[T_PYY] -= bt;
        }
    }
    if (DIR == 0) { bu[1] += ph.colvis * bF[T_PXY]; bu[2] += ph.colvis * bF[T_PXZ]; }
    if (DIR == 1) { bu[0] += ph.colvis * bF[T_PXY]; bu[2] += ph.colvis * bF[T_PYZ]; }
    if (DIR == 2) { bu[0] += ph.colvis * bF[T_PXZ]; bu[1] += ph.colvis * bF[T_PYZ]; }
    bu[DIR] += bun;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        bQ[MX + a] += bu[a] * s.ri;
        bri += bu[a] * Q[MX + a];
    }
    const double smsq = Q[MX] * Q[MX] + Q[MY] * Q[MY] + Q[MZ] * Q[MZ];
    const double Praw = ph.gm1 * (Q[EN] - 0.5 * s.ri * smsq);
    if (!(Praw < ph.P_floor)) {
        bQ[EN] += ph.gm1 * bP;
        bri += -0.5 * ph.gm1 * smsq * bP;
#pragma unroll
        for (int a = 0; a < 3; a++) bQ[MX + a] += -ph.gm1 * s.ri * Q[MX + a] * bP;
    }
    bQ[RH] += -s.ri * s.ri * bri;
}

// reverse of pr::prim and the physical flux of direction DIR: bF (cotangent of F) -> bQ (+=)
template <int NQ, int DIR>
__device__ __forceinline__ void flux_vjp(const Phys& ph, const double* Q, const pr::Prim& s, const double* bF,
                                         double* bQ) {
    if constexpr (NQ == 13) {
        flux13_vjp<DIR>(ph, Q, s, bF, bQ);
        return;
    }
    constexpr int ND = MX + DIR;
    const double un = s.u[DIR];
    double Pn[3] = {0., 0., 0.};
    int pidx[3] = {0, 0, 0};
    if constexpr (NQ == 11) {
        if (DIR == 0) { pidx[0] = PXX; pidx[1] = PXY; pidx[2] = PXZ; }
        if (DIR == 1) { pidx[0] = PXY; pidx[1] = PYY; pidx[2] = PYZ; }
        if (DIR == 2) { pidx[0] = PXZ; pidx[1] = PYZ; pidx[2] = PZZ; }
        Pn[0] = Q[pidx[0]]; Pn[1] = Q[pidx[1]]; Pn[2] = Q[pidx[2]];
    }
    const double P = s.pf;
    double bun = bF[MX] * Q[MX] + bF[MY] * Q[MY] + bF[MZ] * Q[MZ] + bF[EN] * (Q[EN] + P);
    bQ[MX] += bF[MX] * un;
    bQ[MY] += bF[MY] * un;
    bQ[MZ] += bF[MZ] * un;
    bQ[EN] += bF[EN] * un;
    bQ[ND] += bF[RH];
    const double bP = bF[ND] + bF[EN] * un;
    double bu[3] = {bF[EN] * Pn[0], bF[EN] * Pn[1], bF[EN] * Pn[2]};
    if constexpr (NQ == 11) {
#pragma unroll
        for (int a = 0; a < 3; a++) bQ[pidx[a]] += bF[MX + a] + bF[EN] * s.u[a];
        bun += (DIR == 0 ? ph.c4d3cv : -ph.c2d3cv) * bF[PXX] + (DIR == 1 ? ph.c4d3cv : -ph.c2d3cv) * bF[PYY] +
               (DIR == 2 ? ph.c4d3cv : -ph.c2d3cv) * bF[PZZ];
        if (DIR == 0) { bu[1] += ph.colvis * bF[PXY]; bu[2] += ph.colvis * bF[PXZ]; }
        if (DIR == 1) { bu[0] += ph.colvis * bF[PXY]; bu[2] += ph.colvis * bF[PYZ]; }
        if (DIR == 2) { bu[0] += ph.colvis * bF[PXZ]; bu[1] += ph.colvis * bF[PYZ]; }
    }
    bu[DIR] += bun;
    // primitives: u_a = m_a/rho, P = gm1*(E - 0.5/rho*|m|^2) unless floored
    double bri = 0.;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        bQ[MX + a] += bu[a] * s.ri;
        bri += bu[a] * Q[MX + a];
    }
    const double smsq = Q[MX] * Q[MX] + Q[MY] * Q[MY] + Q[MZ] * Q[MZ];
    const double Praw = ph.gm1 * (Q[EN] - 0.5 * s.ri * smsq);
    if (!(Praw < ph.P_floor)) {
        bQ[EN] += ph.gm1 * bP;
        bri += -0.5 * ph.gm1 * smsq * bP;
#pragma unroll
        for (int a = 0; a < 3; a++) bQ[MX + a] += -ph.gm1 * s.ri * Q[MX + a] * bP;
    }
    bQ[RH] += -s.ri * s.ri * bri;
}

// ---------------------------------------------------------------- HLLC ----
// reverse of the HLLC flux for the Euler fields: mu (cotangent of out[0..4])
// -> bQL, bQR (+=, Euler fields), bFL, bFR (+=, Euler fields).  Returns false
// when no branch applied (out kept the central flux).
template <int DIR>
__device__ __forceinline__ bool hllc_vjp(const Phys& ph, const double* QL, const double* QR, const double* mu,
                                         double* bQL, double* bQR, double* bFL, double* bFR) {
    constexpr int IP = MX + DIR, I1 = MX + (DIR + 1) % 3, I2 = MX + (DIR + 2) % 3;
    // the forward flux's own speeds and branch
    const double rL = QL[RH], rR = QR[RH];
    const pr::Side L = pr::side(ph, QL), R = pr::side(ph, QR);
    const pr::HllcSpeeds w = pr::hllc_speeds<DIR>(ph, rL, L, rR, R);
    const double uL = L.u[DIR], uR = R.u[DIR], pL = L.p, pR = R.p;
    const double v2L = L.u[0] * L.u[0] + L.u[1] * L.u[1] + L.u[2] * L.u[2];
    const double v2R = R.u[0] * R.u[0] + R.u[1] * R.u[1] + R.u[2] * R.u[2];
    const double cL = w.cL, cR = w.cR, SL = w.SL, SR = w.SR, SM = w.SM, aR = w.aR, aL = w.aL, sm_den = w.den;
    const bool sl_left = (uL - cL) <= (uR - cR);   // fmin picks uL - cL
    const bool sr_right = (uR + cR) >= (uL + cL);  // fmax picks uR + cR
    const bool den_floor = w.den_floor;
    const int sel = w.sel;
    if (sel < 0) return false;
    if (sel == 0) {
#pragma unroll
        for (int f = 0; f < 5; f++) bFL[f] += mu[f];
        return true;
    }
    if (sel == 3) {
#pragma unroll
        for (int f = 0; f < 5; f++) bFR[f] += mu[f];
        return true;
    }
    const bool left = (sel == 1);
    const double* Qk = left ? QL : QR;
    const double Sk = left ? SL : SR;
    const double uk = left ? uL : uR, pk = left ? pL : pR;
    const double pstar = rL * (uL - SL) * (uL - SM) + pL;
    double den = Sk - SM;
    const bool kden_floor = (den == 0.0);
    if (kden_floor) den = ph.rh_floor;
    const double rid = pr::rcp(den);
    const double sq = Sk - uk;
    const double t1 = sq * Qk[IP] + pstar - pk;
    const double t4 = sq * Qk[EN] - pk * uk + pstar * SM;
    const double s[5] = {Qk[RH] * sq * rid, t1 * rid, sq * Qk[I1] * rid, sq * Qk[I2] * rid, t4 * rid};
    const int fld[5] = {RH, IP, I1, I2, EN};
    // ---- reverse: out[f] = Fk[f] + Sk*(s_f - Qk[f])
    double bQk[5] = {0., 0., 0., 0., 0.};  // indexed like fld
    double bSk = 0., bs[5];
#pragma unroll
    for (int e = 0; e < 5; e++) {
        const double m = mu[fld[e]];
        bSk += m * (s[e] - Qk[fld[e]]);
        bs[e] = m * Sk;
        bQk[e] -= m * Sk;
    }
    double* bFk = left ? bFL : bFR;
#pragma unroll
    for (int f = 0; f < 5; f++) bFk[f] += mu[f];
    double bsq = 0., brid = 0., bpstar = 0., bpk = 0., buk = 0., bSM = 0.;
    // s0 = Qk[RH]*sq*rid
    bQk[0] += bs[0] * sq * rid; bsq += bs[0] * Qk[RH] * rid; brid += bs[0] * Qk[RH] * sq;
    // s1 = t1*rid
    bsq += bs[1] * Qk[IP] * rid; bQk[1] += bs[1] * sq * rid; bpstar += bs[1] * rid; bpk -= bs[1] * rid;
    brid += bs[1] * t1;
    // s2, s3
    bsq += bs[2] * Qk[I1] * rid; bQk[2] += bs[2] * sq * rid; brid += bs[2] * sq * Qk[I1];
    bsq += bs[3] * Qk[I2] * rid; bQk[3] += bs[3] * sq * rid; brid += bs[3] * sq * Qk[I2];
    // s4 = t4*rid
    bsq += bs[4] * Qk[EN] * rid; bQk[4] += bs[4] * sq * rid; bpk -= bs[4] * uk * rid; buk -= bs[4] * pk * rid;
    bpstar += bs[4] * SM * rid; bSM += bs[4] * pstar * rid; brid += bs[4] * t4;
    // rid = 1/den, den = Sk - SM
    if (!kden_floor) {
        const double bden = -brid * rid * rid;
        bSk += bden;
        bSM -= bden;
    }
    // sq = Sk - uk
    bSk += bsq;
    buk -= bsq;
    // pstar = rL*(uL-SL)*(uL-SM) + pL
    double brL = bpstar * (uL - SL) * (uL - SM);
    double buL = bpstar * rL * ((uL - SM) + (uL - SL));
    double bSL = -bpstar * rL * (uL - SM);
    bSM -= bpstar * rL * (uL - SL);
    double bpL = bpstar, bpR = 0., brR = 0., buR = 0., bSR = 0.;
    if (left) { bpL += bpk; buL += buk; bSL += bSk; } else { bpR += bpk; buR += buk; bSR += bSk; }
    // SM = sm_num/sm_den
    const double bnum = bSM / sm_den;
    const double bdenm = den_floor ? 0. : -bSM * SM / sm_den;
    double baR = bnum * uR + bdenm, baL = -bnum * uL - bdenm;
    buR += bnum * aR;
    buL -= bnum * aL;
    bpL += bnum;
    bpR -= bnum;
    // aR = rR*(SR-uR), aL = rL*(SL-uL)
    brR += baR * (SR - uR); bSR += baR * rR; buR -= baR * rR;
    brL += baL * (SL - uL); bSL += baL * rL; buL -= baL * rL;
    // SL = min(uL-cL, uR-cR), SR = max(uR+cR, uL+cL)
    double bcL = 0., bcR = 0.;
    if (sl_left) { buL += bSL; bcL -= bSL; } else { buR += bSL; bcR -= bSL; }
    if (sr_right) { buR += bSR; bcR += bSR; } else { buL += bSR; bcL += bSR; }
    // c = sqrt(gamma*p*ri)
    double briL = 0., briR = 0.;
    if (cL > 0.) { bpL += bcL * ph.gamma * L.ri / (2. * cL); briL += bcL * ph.gamma * pL / (2. * cL); }
    if (cR > 0.) { bpR += bcR * ph.gamma * R.ri / (2. * cR); briR += bcR * ph.gamma * pR / (2. * cR); }
    // scatter the star-state field cotangents onto side k
    double* bQkf = left ? bQL : bQR;
    bQkf[RH] += bQk[0]; bQkf[IP] += bQk[1]; bQkf[I1] += bQk[2]; bQkf[I2] += bQk[3]; bQkf[EN] += bQk[4];
    // p = gm1*(E - 0.5*rho*|u|^2), u_a = m_a*ri, ri = 1/rho; u_dir also enters directly
    {
        double bu[3] = {0., 0., 0.};
        bu[DIR] += buL;
        bQL[EN] += ph.gm1 * bpL;
        brL += -0.5 * ph.gm1 * v2L * bpL;
#pragma unroll
        for (int a = 0; a < 3; a++) bu[a] += -ph.gm1 * rL * L.u[a] * bpL;
#pragma unroll
        for (int a = 0; a < 3; a++) { bQL[MX + a] += bu[a] * L.ri; briL += bu[a] * QL[MX + a]; }
        bQL[RH] += brL - L.ri * L.ri * briL;
    }
    {
        double bu[3] = {0., 0., 0.};
        bu[DIR] += buR;
        bQR[EN] += ph.gm1 * bpR;
        brR += -0.5 * ph.gm1 * v2R * bpR;
#pragma unroll
        for (int a = 0; a < 3; a++) bu[a] += -ph.gm1 * rR * R.u[a] * bpR;
#pragma unroll
        for (int a = 0; a < 3; a++) { bQR[MX + a] += bu[a] * R.ri; briR += bu[a] * QR[MX + a]; }
        bQR[RH] += brR - R.ri * R.ri * briR;
    }
    return true;
}

// The Euler fields of the face flux reversed to the cotangents of both sides'
// physical fluxes (bFL, bFR, set) and of their states through the solver
// (bQL, bQR, +=).
template <int RM, int DIR>
__device__ __forceinline__ void riemann_vjp(const Phys& ph, const double* QL, const double* QR, const double* mu,
                                            double* bQL, double* bQR, double* bFL, double* bFR) {
#pragma unroll
    for (int f = 0; f < 5; f++) { bFL[f] = 0.5 * mu[f]; bFR[f] = 0.5 * mu[f]; }
    if constexpr (RM == RIEMANN_HLLC) {
        double zL[5] = {0., 0., 0., 0., 0.}, zR[5] = {0., 0., 0., 0., 0.};
        if (hllc_vjp<DIR>(ph, QL, QR, mu, bQL, bQR, zL, zR)) {
            // HLLC replaced the central flux of rh..en
#pragma unroll
            for (int f = 0; f < 5; f++) { bFL[f] = zL[f]; bFR[f] = zR[f]; }
        }
    }
    if constexpr (RM == RIEMANN_ROE) {
        // Roe: 0.5 (FL + FR) minus the dissipation of rh..en (or the
        // Lax-Friedrichs fallback); the reverse adds both parts
#pragma unroll
        for (int f = 0; f < 5; f++) { bFL[f] = 0.; bFR[f] = 0.; }
        roe_point_vjp<DIR>(ph, QL, QR, mu, bQL, bQR, bFL, bFR);
    }
}

// face flux reverse: mu (cotangent of the face flux, all fields) -> bQL, bQR (+=)
template <int NQ, int RM, int DIR>
__device__ __forceinline__ void face_vjp(const Phys& ph, const double* QL, const double* QR, const double* mu,
                                         double* bQL, double* bQR) {
    double bFL[NQ], bFR[NQ];
#pragma unroll
    for (int f = 5; f < NQ; f++) { bFL[f] = 0.5 * mu[f]; bFR[f] = 0.5 * mu[f]; }
    riemann_vjp<RM, DIR>(ph, QL, QR, mu, bQL, bQR, bFL, bFR);
    flux_vjp<NQ, DIR>(ph, QL, pr::prim<NQ>(ph, QL), bFL, bQL);
    flux_vjp<NQ, DIR>(ph, QR, pr::prim<NQ>(ph, QR), bFR, bQR);
}

// ------------------------------------------------------------ limiter ----
// The limiter's factors for one cell (the same decisions and values as
// fz::limit_cell): modes >= 2 of rh are scaled by th_rho and then, with the
// other Euler fields, by th_p; `zero` zeroes modes >= 2 of rh..en; `floor`
// also replaces the density average by rh_floor.
struct LimFactors {
    bool floor, zero;
    double th_rho, th_p;
};

template <int NB, int QP, int MQ>
__device__ __forceinline__ LimFactors limit_factors(const double (&m0)[MQ][NB], const LimParams& lp) {
    LimFactors F{false, false, 1.0, 1.0};
    if (m0[RH][0] < lp.rh_floor) {
        F.floor = true;
        F.zero = true;
        return F;
    }
    if (fz::limiter_inactive<NB, MQ>(m0, lp)) return F;
    const auto& T = fz::face_tab<NB>();
    double rho[NB];
#pragma unroll
    for (int r = 0; r < NB; r++) rho[r] = m0[RH][r];
    double rmin = 0.;
#pragma unroll 1
    for (int p = 0; p < 6 * QP * QP; p++) {
        const double* b = T.bf[p / (2 * QP * QP)][(p / (QP * QP)) % 2][p % (QP * QP)];
        double s = 0.;
#pragma unroll
        for (int r = 0; r < NB; r++) s += b[r] * rho[r];
        rmin = (p == 0) ? s : (s < rmin ? s : rmin);
    }
    if (rmin < lp.rh_floor) {
        double theta = (lp.rh_floor - rho[0]) / (rmin - rho[0]);
        if (theta > 1.) theta = 1.;
        if (theta < 0.) theta = 0.;
        F.th_rho = fabs(theta);
#pragma unroll
        for (int r = 1; r < NB; r++) rho[r] = F.th_rho * rho[r];
    }
    const double Pave =
        lp.gm1 * (m0[EN][0] - 0.5 * (m0[MX][0] * m0[MX][0] + m0[MY][0] * m0[MY][0] + m0[MZ][0] * m0[MZ][0]) / rho[0]);
    if (Pave < lp.epsP) {
        F.zero = true;
        return F;
    }
    double pmin = 0.;
#pragma unroll 1
    for (int p = 0; p < 6 * QP * QP; p++) {
        const double* b = T.bf[p / (2 * QP * QP)][(p / (QP * QP)) % 2][p % (QP * QP)];
        double e[5];
#pragma unroll
        for (int f = 0; f < 5; f++) {
            double s = 0.;
#pragma unroll
            for (int r = 0; r < NB; r++) s += b[r] * (f == RH ? rho[r] : m0[f][r]);
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
        F.th_p = theta;
    }
    return F;
}

// cotangent through the frozen limiter, in place
template <int NB, int MQ>
__device__ __forceinline__ void limit_vjp(double (&lam)[MQ][NB], const LimFactors& F) {
    if (F.zero) {
#pragma unroll
        for (int r = 1; r < NB; r++)
#pragma unroll
            for (int f = 0; f < 5; f++) lam[f][r] = 0.0;
        if (F.floor) lam[RH][0] = 0.0;
        return;
    }
#pragma unroll
    for (int r = 1; r < NB; r++) {
        lam[RH][r] *= F.th_rho * F.th_p;
#pragma unroll
        for (int f = 1; f < 5; f++) lam[f][r] *= F.th_p;
    }
}

// ------------------------------------------------------------- stage -----
// three-point rules: grids up to this many cells use the four-wave split of
// the transpose (when its three 64-cell partial sums fit the 160 KB of LDS)
constexpr long kSplitCells = 1L << 17;
template <int NB, int NQ>
constexpr bool split_fits() { return 3L * NQ * NB * 64 * 8 <= 150L * 1024; }

struct AdjParams {
    const double* dt;          // device time step
    double coll;
    double coll_q;             // 13 moments: relaxation rate of the heat flux
    int ivis;
    double a, b;               // out = a*Q^n + b*v
    double bf[3];              // body force
    const double* acc[2];      // lam_in += w[k]*acc[k] (nullptr: none)
    double w[2];
    const double* q_raw;       // stage input before the limiter (nullptr: no limiter)
    LimParams lp;
    const double* out;         // forward stage output and Q^n, for d/dcoll (ivis 1)
    const double* qn;
    double* partial;           // per-block partial sums of d(lam.out)/dcoll
    int rhs_only;              // 1: lam_in = (dR/dm)^T lam (no stage map, no limiter, no sums)
    const double* inflow;      // x-low inflow exterior state (ny,nz,nface,nQ), or nullptr
};

// scale * lam through the transposed relaxation: the stress fields by faci,
// the 13-moment heat flux by faciq
template <int NB, int NQ>
__device__ __forceinline__ void load_lp(const double* __restrict__ lam, const Grid& g, long c, double scale,
                                        double faci, double faciq, double (&l)[NQ][NB]) {
#pragma unroll
    for (int r = 0; r < NB; r++)
#pragma unroll
        for (int f = 0; f < NQ; f++) {
            double v = scale * lam[((long)r * NQ + f) * g.N + c];
            if (NQ == 13 && f >= T_QX) v *= faciq;
            else if (f >= PXX) v *= faci;
            l[f][r] = v;
        }
}

// Lifted cotangent of a face side in face-polynomial form: the transposed
// lift sum_r cf[side][p][r] l_r equals sum_k wb_k(p) L_k with
// L_k = sum over the modes r of pair k of (+-0.25 cb_r Lface_r) l_r.
template <int NB, int NQ, int DIR, int SIDE, int NK>
__device__ __forceinline__ void lift_coeffs(const double (&l)[NQ][NB], double (&L)[NQ][NK]) {
#pragma unroll
    for (int f = 0; f < NQ; f++)
#pragma unroll
        for (int k = 0; k < NK; k++) {
            double s = 0.;
            bool first = true;
#pragma unroll
            for (int r = 0; r < NB; r++) {
                if (fz::pair_index(fz::deg<NB>(r, fz::row_axis(DIR)), fz::deg<NB>(r, fz::col_axis(DIR))) != k) continue;
                constexpr double q = SIDE ? -0.25 : 0.25;
                const double c = q * fz::cbasis<NB>(r) * fz::Lface(fz::deg<NB>(r, DIR), SIDE);
                s = first ? c * l[f][r] : s + c * l[f][r];
                first = false;
            }
            L[f][k] = s;
        }
}

// one face of the cell: adds this cell's share of (dR/dm)^T lp to rt
template <int NB, int QP, int NQ, int RM, int DIR, int SIDE>
__device__ __forceinline__ void face_vjp_cell(const double* __restrict__ q, const double* __restrict__ lam,
                                              const Grid& g, const fz::CellPos& cp, const double (&m)[NQ][NB],
                                              const double (&lo)[NQ][NB], double (&rt)[NQ][NB], const Phys& ph,
                                              double dxi_d, double scale, double faci, double faciq,
                                              const double* __restrict__ inflow) {
    constexpr int NF = QP * QP;
    const auto& T = fz::face_tab<NB>();
    const int n_ax = DIR == 0 ? g.nx : DIR == 1 ? g.ny : g.nz;
    const int a = DIR == 0 ? cp.i : DIR == 1 ? cp.j : cp.k;
    const bool at_edge = SIDE ? (a == n_ax - 1) : (a == 0);
    const int bc = g.bc[2 * DIR + SIDE];
    const bool ext = at_edge && bc != BC_PERIODIC;
    // the neighbour enters through its face polynomial: its trace
    // sum_k kn_k b_k(p) and its lifted cotangent sum_k ln_k wb_k(p), so its
    // modes and cotangents are collapsed as they are loaded
    constexpr int NK = fz::face_nk<NB>();
    const auto& FP = fz::face_poly<NB>();
    double ko[NQ][NK], kn[NQ][NK], ln[NQ][NK];
    // both sides' traces by the forward kernel's functions, so that every
    // Riemann branch is taken as in the forward stage
    sg::signed_coeffs<NB, NQ, DIR, NK>(m, SIDE ? 1.0 : -1.0, ko);
    if (!ext) {
        int an = SIDE ? a + 1 : a - 1;
        if (an < 0) an += n_ax;
        if (an >= n_ax) an -= n_ax;
        const long cn = DIR == 0 ? (cp.c - cp.i + an)
                      : DIR == 1 ? (cp.c + (long)(an - cp.j) * g.nx)
                                 : (cp.c + (long)(an - cp.k) * g.nx * g.ny);
        double nm[NQ][NB], nl[NQ][NB];
        fz::load_modes<NB, NQ>(q, g, cn, nm);
        sg::signed_coeffs<NB, NQ, DIR, NK>(nm, SIDE ? -1.0 : 1.0, kn);
        load_lp<NB, NQ>(lam, g, cn, scale, faci, faciq, nl);
        lift_coeffs<NB, NQ, DIR, 1 - SIDE, NK>(nl, ln);
    }
    bool zero_normal = false;
    if (ext && bc == BC_OUTFLOW && !(DIR == 0 && SIDE == 1)) {
        double v = 0.;
        for (int p = 0; p < NF; p++) {
            const double s = sg::eval_one<NK>(ko[MX + DIR], FP.b[p]);
            v = (p == 0) ? s : (SIDE ? fmin(v, s) : fmax(v, s));
        }
        zero_normal = SIDE ? (v < 0.0) : (v > 0.0);
    }
#pragma unroll 1
    for (int p = 0; p < NF; p++) {
        double own[NQ], oth[NQ], mu[NQ];
        sg::eval_point<NQ, NK>(ko, FP.b[p], own);
#pragma unroll
        for (int f = 0; f < NQ; f++) {
            double t = 0.;
#pragma unroll
            for (int r = 0; r < NB; r++) t += T.cf[DIR][SIDE][p][r] * lo[f][r];
            mu[f] = t;
        }
        bool flip_mx = false;
        if (!ext) {
            sg::eval_point<NQ, NK>(kn, FP.b[p], oth);
#pragma unroll
            for (int f = 0; f < NQ; f++) {
                double t = ln[f][0] * FP.wb[p][0];
#pragma unroll
                for (int k = 1; k < NK; k++) t += ln[f][k] * FP.wb[p][k];
                mu[f] += t;
            }
        } else {
#pragma unroll
            for (int f = 0; f < NQ; f++) oth[f] = own[f];
            if (bc == BC_NOSLIP) {
                oth[MX] = oth[MY] = oth[MZ] = 0.0;
            } else if (bc == BC_WALL) {
                oth[MX + DIR] = 0.0;
            } else if (bc == BC_OUTFLOW) {
                if (DIR == 0 && SIDE == 1) {
                    if (oth[MX] > 0.0) { oth[MX] = -own[MX]; flip_mx = true; }
                } else if (zero_normal) {
                    oth[MX + DIR] = 0.0;
                }
            }
            if constexpr (DIR == 0 && SIDE == 0) {
                if (bc == BC_INFLOW) fz::inflow_ghost<NQ>(inflow, g, cp, p, NF, oth);
            }
        }
#pragma unroll
        for (int f = 0; f < NQ; f++) mu[f] *= dxi_d;
        double bL[NQ], bR[NQ];
#pragma unroll
        for (int f = 0; f < NQ; f++) { bL[f] = 0.; bR[f] = 0.; }
        const double* QL = SIDE ? own : oth;
        const double* QR = SIDE ? oth : own;
        face_vjp<NQ, RM, DIR>(ph, QL, QR, mu, bL, bR);
        double* bo = SIDE ? bL : bR;
        const double* bt = SIDE ? bR : bL;
        if (ext) {
            // ghost = G(own): add G^T of the ghost's cotangent
#pragma unroll
            for (int f = 0; f < NQ; f++) {
                double gcoef = 1.0;
                if (bc == BC_NOSLIP && (f == MX || f == MY || f == MZ)) gcoef = 0.0;
                if (bc == BC_WALL && f == MX + DIR) gcoef = 0.0;
                if (bc == BC_INFLOW && f <= EN) gcoef = 0.0;   // prescribed: no dependence on the interior
                if (bc == BC_OUTFLOW) {
                    if (DIR == 0 && SIDE == 1) {
                        if (f == MX && flip_mx) gcoef = -1.0;
                    } else if (zero_normal && f == MX + DIR) {
                        gcoef = 0.0;
                    }
                }
                bo[f] += gcoef * bt[f];
            }
        }
#pragma unroll
        for (int f = 0; f < NQ; f++) {
            const double v = bo[f];
#pragma unroll
            for (int r = 0; r < NB; r++) rt[f][r] += T.bf[DIR][SIDE][p][r] * v;
        }
    }
}

template <int NB, int QP, int NQ>
__device__ __forceinline__ void volume_vjp(const double (&m)[NQ][NB], const double (&lo)[NQ][NB], double (&rt)[NQ][NB],
                                           const Phys& ph, double dxi, double dyi, double dzi) {
#pragma unroll
    for (int i = 0; i < QP; i++)
#pragma unroll
        for (int j = 0; j < QP; j++)
#pragma unroll
            for (int k = 0; k < QP; k++) {
                double Qp[NQ], mx[NQ], my[NQ], mz[NQ];
#pragma unroll
                for (int f = 0; f < NQ; f++) {
                    double s = 0., ax = 0., ay = 0., az = 0.;
#pragma unroll
                    for (int r = 0; r < NB; r++) {
                        const double b = fz::phi_int<NB, QP>(r, i, j, k);
                        if (b != 0.0) s += b * m[f][r];
                        const double cx = fz::cvol<NB, QP>(0, r, i, j, k);
                        const double cy = fz::cvol<NB, QP>(1, r, i, j, k);
                        const double cz = fz::cvol<NB, QP>(2, r, i, j, k);
                        if (r > 0 && cx != 0.0) ax += cx * lo[f][r];
                        if (r > 0 && cy != 0.0) ay += cy * lo[f][r];
                        if (r > 0 && cz != 0.0) az += cz * lo[f][r];
                    }
                    Qp[f] = s;
                    mx[f] = dxi * ax;
                    my[f] = dyi * ay;
                    mz[f] = dzi * az;
                }
                const pr::Prim st = pr::prim<NQ>(ph, Qp);
                double bQ[NQ];
#pragma unroll
                for (int f = 0; f < NQ; f++) bQ[f] = 0.;
                flux_vjp<NQ, 0>(ph, Qp, st, mx, bQ);
                flux_vjp<NQ, 1>(ph, Qp, st, my, bQ);
                flux_vjp<NQ, 2>(ph, Qp, st, mz, bQ);
#pragma unroll
                for (int f = 0; f < NQ; f++)
#pragma unroll
                    for (int r = 0; r < NB; r++) {
                        const double b = fz::phi_int<NB, QP>(r, i, j, k);
                        if (b != 0.0) rt[f][r] += b * bQ[f];
                    }
                fz::point_barrier();
            }
}

// Parts of the transpose of one cell: bit 0 volume + sources, bits 1..3 the
// x, y, z face pairs.  Adds to rt; returns the cell's share of d/dcoll.
template <int NB, int QP, int NQ, int RM>
__device__ __forceinline__ double cell_vjp_parts(int parts, const double* __restrict__ q,
                                                 const double* __restrict__ lam, const Grid& g, const Phys& ph,
                                                 const AdjParams& ap, const fz::CellPos& cp, double dt, double faci,
                                                 double faciq, const double (&m)[NQ][NB], const double (&lo)[NQ][NB],
                                                 double (&rt)[NQ][NB]) {
    double dcoll = 0.;
    const long c = cp.c;
    if (parts & 1) {
        volume_vjp<NB, QP, NQ>(m, lo, rt, ph, g.dxi, g.dyi, g.dzi);
        fz::fence();
        // sources: ivis 0 explicit relaxation -coll*P; body force rho*g, m.g
        if constexpr (NQ >= 11) {
            // the stress fields (and, with 13 moments, the heat flux at its own rate)
            constexpr int SLAST = NQ == 13 ? T_PYZ : PYZ;
            if (ap.ivis == 0 && ap.coll != 0.) {
#pragma unroll
                for (int f = PXX; f <= SLAST; f++)
#pragma unroll
                    for (int r = 0; r < NB; r++) {
                        rt[f][r] += -ap.coll * lo[f][r];
                        dcoll += -dt * lo[f][r] * m[f][r];
                    }
            }
            if constexpr (NQ == 13) {
                if (ap.ivis == 0 && ap.coll_q != 0.) {
#pragma unroll
                    for (int f = T_QX; f <= T_QZ; f++)
#pragma unroll
                        for (int r = 0; r < NB; r++) rt[f][r] += -ap.coll_q * lo[f][r];
                }
            }
            if (ap.ivis == 1 && ap.coll != 0. && ap.out) {
                // v = faci*(m + dt*R): dv/dcoll = -dt*faci*v, b*v = out - a*Q^n;
                // the branch on a stays outside the element loop so that the
                // loads are issued together
                if (ap.a != 0.) {
#pragma unroll
                    for (int f = PXX; f <= SLAST; f++)
#pragma unroll
                        for (int r = 0; r < NB; r++) {
                            const long o = ((long)r * NQ + f) * g.N + c;
                            const double bv = ap.out[o] - ap.a * ap.qn[o];
                            dcoll += -dt * faci * lam[o] * bv;
                        }
                } else {
#pragma unroll
                    for (int f = PXX; f <= SLAST; f++)
#pragma unroll
                        for (int r = 0; r < NB; r++) {
                            const long o = ((long)r * NQ + f) * g.N + c;
                            const double bv = ap.out[o] - 0.;
                            dcoll += -dt * faci * lam[o] * bv;
                        }
                }
            }
        }
        if (ap.bf[0] != 0. || ap.bf[1] != 0. || ap.bf[2] != 0.) {
#pragma unroll
            for (int r = 0; r < NB; r++) {
                rt[RH][r] += ap.bf[0] * lo[MX][r] + ap.bf[1] * lo[MY][r] + ap.bf[2] * lo[MZ][r];
                rt[MX][r] += ap.bf[0] * lo[EN][r];
                rt[MY][r] += ap.bf[1] * lo[EN][r];
                rt[MZ][r] += ap.bf[2] * lo[EN][r];
            }
        }
    }
    if (parts & 2) {
        face_vjp_cell<NB, QP, NQ, RM, 0, 0>(q, lam, g, cp, m, lo, rt, ph, g.dxi, ap.b, faci, faciq, ap.inflow);
        fz::fence();
        face_vjp_cell<NB, QP, NQ, RM, 0, 1>(q, lam, g, cp, m, lo, rt, ph, g.dxi, ap.b, faci, faciq, ap.inflow);
        fz::fence();
    }
    if (parts & 4) {
        face_vjp_cell<NB, QP, NQ, RM, 1, 0>(q, lam, g, cp, m, lo, rt, ph, g.dyi, ap.b, faci, faciq, ap.inflow);
        fz::fence();
        face_vjp_cell<NB, QP, NQ, RM, 1, 1>(q, lam, g, cp, m, lo, rt, ph, g.dyi, ap.b, faci, faciq, ap.inflow);
        fz::fence();
    }
    if (parts & 8) {
        face_vjp_cell<NB, QP, NQ, RM, 2, 0>(q, lam, g, cp, m, lo, rt, ph, g.dzi, ap.b, faci, faciq, ap.inflow);
        fz::fence();
        face_vjp_cell<NB, QP, NQ, RM, 2, 1>(q, lam, g, cp, m, lo, rt, ph, g.dzi, ap.b, faci, faciq, ap.inflow);
        fz::fence();
    }
    return dcoll;
}

// lam_in = sum_k w_k acc_k + L'^T (lo + dt*rt), or rt alone in rhs mode
template <int NB, int QP, int NQ>
__device__ __forceinline__ void cell_vjp_finish(double* __restrict__ lam_in, const Grid& g, const AdjParams& ap,
                                                long c, double dt, const double (&lo)[NQ][NB], double (&rt)[NQ][NB]) {
    if (ap.rhs_only) {
#pragma unroll
        for (int f = 0; f < NQ; f++)
#pragma unroll
            for (int r = 0; r < NB; r++) lam_in[((long)r * NQ + f) * g.N + c] = rt[f][r];
        return;
    }
#pragma unroll
    for (int f = 0; f < NQ; f++)
#pragma unroll
        for (int r = 0; r < NB; r++) rt[f][r] = lo[f][r] + dt * rt[f][r];
    // each accumulated term under one branch, its values loaded together
#pragma unroll
    for (int t = 0; t < 2; t++) {
        if (ap.acc[t]) {
            double av[NQ][NB];
            fz::load_modes<NB, NQ>(ap.acc[t], g, c, av);
#pragma unroll
            for (int f = 0; f < NQ; f++)
#pragma unroll
                for (int r = 0; r < NB; r++) rt[f][r] += ap.w[t] * av[f][r];
        }
    }
    if (ap.q_raw) {
        double raw[NQ][NB];
        fz::load_modes<NB, NQ>(ap.q_raw, g, c, raw);
        const LimFactors F = limit_factors<NB, QP, NQ>(raw, ap.lp);
        limit_vjp<NB, NQ>(rt, F);
    }
#pragma unroll
    for (int f = 0; f < NQ; f++)
#pragma unroll
        for (int r = 0; r < NB; r++) lam_in[((long)r * NQ + f) * g.N + c] = rt[f][r];
}

// per-block partial of d(lam.out)/dcoll (every thread of the block calls it)
__device__ __forceinline__ void block_partial(double v, double* partial) {
    __shared__ double red[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) s += red[w];
        partial[blockIdx.x] = s;
    }
}

__device__ __forceinline__ fz::CellPos cell_pos(const Grid& g, long c) {
    fz::CellPos cp;
    cp.c = c;
    cp.i = (int)(c % g.nx);
    cp.j = (int)((c / g.nx) % g.ny);
    cp.k = (int)(c / ((long)g.nx * g.ny));
    return cp;
}

// One thread per cell.
template <int NB, int QP, int NQ, int RM>
__global__ __launch_bounds__(256) void k_stage_vjp(const double* __restrict__ q, const double* __restrict__ lam,
                                                   double* __restrict__ lam_in, Grid g, Phys ph, AdjParams ap) {
    const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double dcoll = 0.;
    if (c < g.N) {
        const fz::CellPos cp = cell_pos(g, c);
        const double dt = *ap.dt;
        const double faci = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll) : 1.0;
        const double faciq = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll_q) : 1.0;
        double m[NQ][NB], lo[NQ][NB], rt[NQ][NB];
        fz::load_modes<NB, NQ>(q, g, c, m);
        load_lp<NB, NQ>(lam, g, c, ap.b, faci, faciq, lo);
#pragma unroll
        for (int f = 0; f < NQ; f++)
#pragma unroll
            for (int r = 0; r < NB; r++) rt[f][r] = 0.;
        dcoll = cell_vjp_parts<NB, QP, NQ, RM>(15, q, lam, g, ph, ap, cp, dt, faci, faciq, m, lo, rt);
        cell_vjp_finish<NB, QP, NQ>(lam_in, g, ap, c, dt, lo, rt);
    }
    if (ap.partial) block_partial(dcoll, ap.partial);
}

// For small grids (latency-bound): a block of 4 waves takes 64 cells and each
// wave one part (volume + sources, x, y, z faces); the face waves pass their
// sums through LDS to the volume wave, which finishes the cells.  Four times
// the parallelism of one thread per cell, at the same total work.
template <int NB, int QP, int NQ, int RM>
__global__ __launch_bounds__(256) void k_stage_vjp_split(const double* __restrict__ q,
                                                         const double* __restrict__ lam, double* __restrict__ lam_in,
                                                         Grid g, Phys ph, AdjParams ap) {
    static_assert(split_fits<NB, NQ>(), "partial sums exceed LDS");
    __shared__ double part_sum[3][NQ * NB][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long c = (long)blockIdx.x * 64 + lane;
    double dcoll = 0.;
    const double dt = *ap.dt;
    const double faci = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll) : 1.0;
    const double faciq = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll_q) : 1.0;
    double m[NQ][NB], lo[NQ][NB], rt[NQ][NB];
#pragma unroll
    for (int f = 0; f < NQ; f++)
#pragma unroll
        for (int r = 0; r < NB; r++) rt[f][r] = 0.;
    const bool valid = c < g.N;
    fz::CellPos cp;
    if (valid) {
        cp = cell_pos(g, c);
        fz::load_modes<NB, NQ>(q, g, c, m);
        load_lp<NB, NQ>(lam, g, c, ap.b, faci, faciq, lo);
        dcoll = cell_vjp_parts<NB, QP, NQ, RM>(1 << wave, q, lam, g, ph, ap, cp, dt, faci, faciq, m, lo, rt);
    }
    if (wave > 0) {
#pragma unroll
        for (int f = 0; f < NQ; f++)
#pragma unroll
            for (int r = 0; r < NB; r++) part_sum[wave - 1][f * NB + r][lane] = rt[f][r];
    }
    __syncthreads();
    if (wave == 0 && valid) {
#pragma unroll
        for (int f = 0; f < NQ; f++)
#pragma unroll
            for (int r = 0; r < NB; r++)
                rt[f][r] += part_sum[0][f * NB + r][lane] + part_sum[1][f * NB + r][lane] +
                            part_sum[2][f * NB + r][lane];
        cell_vjp_finish<NB, QP, NQ>(lam_in, g, ap, c, dt, lo, rt);
    }
    if (ap.partial) block_partial(dcoll, ap.partial);
}

// ------------------------------------------- a point, then a field a lane ----
// One volume point of a cell whose modes and cotangents lie in LDS (field f at
// m + f*fs, lo + f*fs): its state, the cotangents of its three fluxes (the
// transposes of the volume sums; b: the basis there, w: 0.25 times its weight)
// and the fluxes reversed to the state's cotangent bQ.
template <int NB, int NQ>
__device__ __forceinline__ void volume_point_vjp(const double* m, const double* lo, int fs,
                                                 const double* __restrict__ bp, double w, const Grid& g,
                                                 const Phys& ph, double (&bQ)[NQ]) {
    double b[NB], Qp[NQ], bF[NQ];
#pragma unroll
    for (int r = 0; r < NB; r++) b[r] = bp[r];
#pragma unroll
    for (int f = 0; f < NQ; f++) {
        double v = m[f * fs];
#pragma unroll
        for (int r = 1; r < NB; r++) v += b[r] * m[f * fs + r];
        Qp[f] = v;
        bQ[f] = 0.;
    }
    const pr::Prim st = pr::prim<NQ>(ph, Qp);
    const double h[3] = {g.dxi * w, g.dyi * w, g.dzi * w};
    // cotangent of a field's flux: sum_r cb_r d(phi_r) lo_r
#pragma unroll
    for (int f = 0; f < NQ; f++) {
        const double* const l = lo + f * fs;
        double s = 3. * l[KX];
        if constexpr (NB > 4) s += 9. * b[KZ] * l[KZX] + 9. * b[KY] * l[KXY];
        if constexpr (NB == 10) s += 15. * b[KX] * l[KXX];
        if constexpr (NB == 8) s += 27. * b[KYZ] * l[KXYZ];
        bF[f] = h[0] * s;
    }
    flux_vjp<NQ, 0>(ph, Qp, st, bF, bQ);
    sg::section();
#pragma unroll
    for (int f = 0; f < NQ; f++) {
        const double* const l = lo + f * fs;
        double s = 3. * l[KY];
        if constexpr (NB > 4) s += 9. * b[KZ] * l[KYZ] + 9. * b[KX] * l[KXY];
        if constexpr (NB == 10) s += 15. * b[KY] * l[KYY];
        if constexpr (NB == 8) s += 27. * b[KZX] * l[KXYZ];
        bF[f] = h[1] * s;
    }
    flux_vjp<NQ, 1>(ph, Qp, st, bF, bQ);
    sg::section();
#pragma unroll
    for (int f = 0; f < NQ; f++) {
        const double* const l = lo + f * fs;
        double s = 3. * l[KZ];
        if constexpr (NB > 4) s += 9. * b[KY] * l[KYZ] + 9. * b[KX] * l[KZX];
        if constexpr (NB == 10) s += 15. * b[KZ] * l[KZZ];
        if constexpr (NB == 8) s += 27. * b[KXY] * l[KXYZ];
        bF[f] = h[2] * s;
    }
    flux_vjp<NQ, 2>(ph, Qp, st, bF, bQ);
}

// Field f of cell c from the sum rt of its face and volume terms: the sources,
// the stage map (lo + dt*rt, the accumulated terms) and the frozen limiter
// (zero, floor: bits of `lim`), as cell_vjp_parts and cell_vjp_finish, stored;
// returns the field's share of d/dcoll.  m: this field's modes, lo: the cell's
// cotangents, field e at lo + e*fs.
template <int NB, int NQ>
__device__ __forceinline__ double field_finish(const double* __restrict__ lam, double* __restrict__ lam_in,
                                               const Grid& g, const AdjParams& ap, int f, long c, double dt,
                                               double faci, const double* m, const double* lo, int fs, int lim,
                                               double th_rho, double th_p, double (&rt)[NB]) {
    double dcoll = 0.;
    double lof[NB];
#pragma unroll
    for (int r = 0; r < NB; r++) lof[r] = lo[f * fs + r];
    if constexpr (NQ >= 11) {
        constexpr int SLAST = NQ == 13 ? T_PYZ : PYZ;
        if (ap.ivis == 0) {
            if (f >= PXX && f <= SLAST && ap.coll != 0.)
#pragma unroll
                for (int r = 0; r < NB; r++) {
                    rt[r] += -ap.coll * lof[r];
                    dcoll += -dt * lof[r] * m[r];
                }
            if (NQ == 13 && f >= T_QX && ap.coll_q != 0.)
#pragma unroll
                for (int r = 0; r < NB; r++) rt[r] += -ap.coll_q * lof[r];
        }
        if (ap.ivis == 1 && ap.coll != 0. && ap.out && f >= PXX && f <= SLAST) {
            // qn is read only when its weight a is nonzero (callers pass no
            // qn for the first stage)
            const bool with_qn = ap.a != 0.;
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const long o = qoff(g, c, f, r);
                const double bv = with_qn ? ap.out[o] - ap.a * ap.qn[o] : ap.out[o];
                dcoll += -dt * faci * lam[o] * bv;
            }
        }
    }
    if (ap.bf[0] != 0. || ap.bf[1] != 0. || ap.bf[2] != 0.) {
        // lo of the Euler fields (relaxation factor 1)
        if (f == RH)
#pragma unroll
            for (int r = 0; r < NB; r++)
                rt[r] += ap.bf[0] * lo[MX * fs + r] + ap.bf[1] * lo[MY * fs + r] + ap.bf[2] * lo[MZ * fs + r];
        if (f >= MX && f <= MZ) {
            const double bf = f == MX ? ap.bf[0] : (f == MY ? ap.bf[1] : ap.bf[2]);
#pragma unroll
            for (int r = 0; r < NB; r++) rt[r] += bf * lo[EN * fs + r];
        }
    }
    if (!ap.rhs_only) {
#pragma unroll
        for (int r = 0; r < NB; r++) rt[r] = lof[r] + dt * rt[r];
#pragma unroll
        for (int e = 0; e < 2; e++)
            if (ap.acc[e])
#pragma unroll
                for (int r = 0; r < NB; r++) rt[r] += ap.w[e] * ap.acc[e][qoff(g, c, f, r)];
        if (ap.q_raw && f <= EN) {
            if (lim & 1) {
#pragma unroll
                for (int r = 1; r < NB; r++) rt[r] = 0.0;
                if ((lim & 2) && f == RH) rt[0] = 0.0;
            } else {
                const double th = f == RH ? th_rho * th_p : th_p;
#pragma unroll
                for (int r = 1; r < NB; r++) rt[r] *= th;
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NB; r++) lam_in[qoff(g, c, f, r)] = rt[r];
    return dcoll;
}

// the limiter's factors of cell c, for field_finish
template <int NB, int QP>
__device__ __forceinline__ void limit_terms(const AdjParams& ap, const Grid& g, long c, int& lim, double& th_rho,
                                            double& th_p) {
    double raw[5][NB];
#pragma unroll
    for (int e = 0; e < 5; e++)
#pragma unroll
        for (int r = 0; r < NB; r++) raw[e][r] = ap.q_raw[qoff(g, c, e, r)];
    const LimFactors L = limit_factors<NB, QP, 5>(raw, ap.lp);
    th_rho = L.th_rho;
    th_p = L.th_p;
    lim = (L.zero ? 1 : 0) + (L.floor ? 2 : 0);
}

// per-block partial of d(lam.out)/dcoll for workgroups of W waves
template <int W>
__device__ __forceinline__ void block_partial_of(double v, double* partial) {
    __shared__ double red[W];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.;
        for (int w = 0; w < W; w++) s += red[w];
        partial[blockIdx.x] = s;
    }
}

// Two-point rules (nbasis 4 and 8): a workgroup of eight waves takes 16 cells,
// each of its first six waves one face of each (a lane a face point: 16 cells
// by 4 points), the last two the volume points.  The cells' own modes and
// cotangents lie in LDS for all; a face wave adds its neighbours' face
// coefficients.  Then a field of a cell a lane sums the points and finishes.
// Bound by latency (a chain of loads, one point, the sums) on the grids it is
// for; five fields run as fast in 128 registers, two workgroups a CU (64,000
// cells: 71 us against 96 with 256), more fields spill there (8,192 cells, 11
// fields: 22.4 us against 20.8 with 256).
constexpr int kPointCells = 16;

template <int NB, int NQ, int DIR, int SIDE>
__device__ __forceinline__ bool face_neighbour(const Grid& g, long c, long& cn) {
    const long sd = DIR == 0 ? 1 : DIR == 1 ? g.nx : (long)g.nx * g.ny;
    const int n_ax = DIR == 0 ? g.nx : DIR == 1 ? g.ny : g.nz;
    const int a = (int)(DIR == 0 ? c % g.nx : DIR == 1 ? (c / g.nx) % g.ny : c / ((long)g.nx * g.ny));
    const bool edge = SIDE ? a == n_ax - 1 : a == 0;
    cn = SIDE ? (edge ? c - (n_ax - 1) * sd : c + sd) : (edge ? c + (n_ax - 1) * sd : c - sd);
    return edge && g.bc[2 * DIR + SIDE] != BC_PERIODIC;  // a boundary face: cn is not its neighbour
}

// trace and lifted-cotangent coefficients of the neighbours, to kn
template <int NB, int NQ, int DIR, int SIDE>
__device__ __forceinline__ void load_neighbours(double* kn, const double* __restrict__ q,
                                                const double* __restrict__ lam, long c0, const Grid& g,
                                                double b, double faci, double faciq) {
    constexpr int NK = fz::face_nk<NB>(), C = kPointCells;
    const int lane = (int)(threadIdx.x & 63);
    const long c = c0 + lane % C < g.N ? c0 + lane % C : g.N - 1;
    long cn;
    if (face_neighbour<NB, NQ, DIR, SIDE>(g, c, cn)) return;
#pragma unroll
    for (int n = 0; n < (NQ * C + 63) / 64; n++) {
        const int it = lane + 64 * n, f = it / C;
        if (it < NQ * C) {
            double m[1][NB], l[1][NB], K[1][NK], L[1][NK];
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const long o = ((long)r * NQ + f) * g.N + cn;
                m[0][r] = q[o];
                l[0][r] = lam[o];
            }
            sg::signed_coeffs<NB, 1, DIR, NK>(m, SIDE ? -1.0 : 1.0, K);
            lift_coeffs<NB, 1, DIR, 1 - SIDE, NK>(l, L);
            const double fac = b * (NQ == 13 && f >= T_QX ? faciq : (f >= PXX ? faci : 1.0));
#pragma unroll
            for (int k = 0; k < NK; k++) {
                kn[it * NK + k] = K[0][k];
                kn[(NQ * C + it) * NK + k] = fac * L[0][k];
            }
        }
    }
}

// One face point of a cell: the cotangent of the cell's trace to the wave's
// part of LDS (kn, its neighbours' coefficients until then).
template <int NB, int QP, int NQ, int RM, int DIR, int SIDE>
__device__ __forceinline__ void face_point_vjp(double* kn, const double* m_s, const double* lo_s, long c0,
                                               const Grid& g, const Phys& ph, const double* __restrict__ inflow) {
    constexpr int NF = QP * QP, NK = fz::face_nk<NB>(), C = kPointCells;
    static_assert(NF * C == 64, "a wave is 16 cells by 4 points");
    const auto& FP = fz::face_poly<NB>();
    const int lane = (int)(threadIdx.x & 63), p = lane / C, lc = lane % C;
    const long c = c0 + lc < g.N ? c0 + lc : g.N - 1;
    long cn;
    const bool ext = face_neighbour<NB, NQ, DIR, SIDE>(g, c, cn);
    const int bc = g.bc[2 * DIR + SIDE];
    const double dxi_d = DIR == 0 ? g.dxi : DIR == 1 ? g.dyi : g.dzi;
    double b[NK], wb[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        b[k] = FP.b[p][k];
        wb[k] = dxi_d * FP.wb[p][k];
    }
    // field f of the cell's trace (by the forward kernel's functions, so that
    // every Riemann branch is taken as in the forward stage), of the
    // neighbour's, and of the flux's cotangent
    auto own_at = [&](int f) {
        double m[1][NB], K[1][NK];
#pragma unroll
        for (int r = 0; r < NB; r++) m[0][r] = m_s[(f * C + lc) * NB + r];
        sg::signed_coeffs<NB, 1, DIR, NK>(m, SIDE ? 1.0 : -1.0, K);
        return sg::eval_one<NK>(K[0], b);
    };
    auto other_at = [&](int f) {
        return sg::eval_one<NK>(kn + (f * C + lc) * NK, b);
    };
    auto mu_at = [&](int f) {
        double l[1][NB], L[1][NK];
#pragma unroll
        for (int r = 0; r < NB; r++) l[0][r] = lo_s[(f * C + lc) * NB + r];
        lift_coeffs<NB, 1, DIR, SIDE, NK>(l, L);
        const double* const k = kn + (NQ * C + f * C + lc) * NK;
        double s = 0.;
#pragma unroll
        for (int e = 0; e < NK; e++) s += (ext ? L[0][e] : L[0][e] + k[e]) * wb[e];
        return s;
    };
    double own[NQ], oth[NQ], mu[NQ], bo[NQ], bt[NQ], bFo[NQ], bFt[NQ];
#pragma unroll
    for (int f = 0; f < NQ; f++) {
        bo[f] = 0.;
        bt[f] = 0.;
    }
#pragma unroll
    for (int f = 0; f < 5; f++) {
        own[f] = own_at(f);
        mu[f] = mu_at(f);
    }
    bool zero_normal = false, flip_mx = false;
    if (ext) {
#pragma unroll
        for (int f = 0; f < 5; f++) oth[f] = own[f];
        if (bc == BC_NOSLIP) {
            oth[MX] = oth[MY] = oth[MZ] = 0.0;
        } else if (bc == BC_WALL) {
            oth[MX + DIR] = 0.0;
        } else if (bc == BC_OUTFLOW) {
            if (DIR == 0 && SIDE == 1) {
                if (oth[MX] > 0.0) { oth[MX] = -own[MX]; flip_mx = true; }
            } else {
                // the face's extreme normal momentum decides for all its points
                double v = own[MX + DIR];
#pragma unroll
                for (int o = C; o < 64; o <<= 1) {
                    const double w = __shfl_xor(v, o, 64);
                    v = SIDE ? fmin(v, w) : fmax(v, w);
                }
                zero_normal = SIDE ? (v < 0.0) : (v > 0.0);
                if (zero_normal) oth[MX + DIR] = 0.0;
            }
        }
        if constexpr (DIR == 0 && SIDE == 0) {
            if (bc == BC_INFLOW) {
                fz::CellPos cp;
                cp.c = c;
                cp.i = 0;
                cp.j = (int)((c / g.nx) % g.ny);
                cp.k = (int)(c / ((long)g.nx * g.ny));
                fz::inflow_ghost<NQ>(inflow, g, cp, p, NF, oth);
            }
        }
    } else {
#pragma unroll
        for (int f = 0; f < 5; f++) oth[f] = other_at(f);
    }
    // face_vjp in parts (the Riemann solver's Euler fields, the cell's own
    // flux, at a boundary the ghost's), so that no part holds all that the
    // point has
    riemann_vjp<RM, DIR>(ph, SIDE ? own : oth, SIDE ? oth : own, mu, SIDE ? bo : bt, SIDE ? bt : bo,
                         SIDE ? bFo : bFt, SIDE ? bFt : bFo);
    sg::section();
#pragma unroll
    for (int f = 5; f < NQ; f++) {
        own[f] = own_at(f);
        bFo[f] = 0.5 * mu_at(f);
    }
    flux_vjp<NQ, DIR>(ph, own, pr::prim<NQ>(ph, own), bFo, bo);
    sg::section();
    if (ext) {
        // ghost = G(own): add G^T of the ghost's cotangent
#pragma unroll
        for (int f = 5; f < NQ; f++) {
            oth[f] = own_at(f);
            bFt[f] = 0.5 * mu_at(f);
        }
        flux_vjp<NQ, DIR>(ph, oth, pr::prim<NQ>(ph, oth), bFt, bt);
#pragma unroll
        for (int f = 0; f < NQ; f++) {
            double gcoef = 1.0;
            if (bc == BC_NOSLIP && (f == MX || f == MY || f == MZ)) gcoef = 0.0;
            if (bc == BC_WALL && f == MX + DIR) gcoef = 0.0;
            if (bc == BC_INFLOW && f <= EN) gcoef = 0.0;  // prescribed: no dependence on the interior
            if (bc == BC_OUTFLOW) {
                if (DIR == 0 && SIDE == 1) {
                    if (f == MX && flip_mx) gcoef = -1.0;
                } else if (zero_normal && f == MX + DIR) {
                    gcoef = 0.0;
                }
            }
            bo[f] += gcoef * bt[f];
        }
    }
    sg::section();  // the wave has read its neighbours' coefficients
#pragma unroll
    for (int f = 0; f < NQ; f++) kn[f * 64 + lane] = bo[f];
}

template <int NB, int QP, int NQ, int RM>
__global__ __launch_bounds__(512, (NQ == 5 ? 4 : 2)) void k_points_vjp(const double* __restrict__ q, const double* __restrict__ lam,
                                                       double* __restrict__ lam_in, const Tables* __restrict__ T,
                                                       Grid g, Phys ph, AdjParams ap) {
    constexpr int NK = fz::face_nk<NB>(), C = kPointCells, NPG = QP * QP * QP, NF = QP * QP;
    static_assert(NPG * C == 128, "two waves of volume points");
    __shared__ __attribute__((aligned(16))) double m_s[NQ * C * NB], lo_s[NQ * C * NB];
    __shared__ __attribute__((aligned(16))) double kn_s[6][2 * NQ * C * NK];
    __shared__ double bq_s[NQ][NPG * C];
    __shared__ double th_s[2][C];
    __shared__ int lim_s[C];
    const int t = (int)threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const long c0 = (long)xcd_block() * C;
    const double dt = *ap.dt;
    const double faci = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll) : 1.0;
    const double faciq = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll_q) : 1.0;
#pragma unroll
    for (int n = 0; n < (NQ * NB * C + 511) / 512; n++) {
        const int it = t + n * 512;
        if (it < NQ * NB * C) {
            const int c = it % C, row = it / C, r = row / NQ, f = row % NQ;
            // lanes past the grid take a copy of the last cell and store nothing
            const long o = (long)row * g.N + (c0 + c < g.N ? c0 + c : g.N - 1);
            m_s[(f * C + c) * NB + r] = q[o];
            lo_s[(f * C + c) * NB + r] = ap.b * lam[o] * (NQ == 13 && f >= T_QX ? faciq : (f >= PXX ? faci : 1.0));
        }
    }
    double* const kn = kn_s[wave < 6 ? wave : 0];
    switch (wave) {
    case 0: load_neighbours<NB, NQ, 0, 0>(kn, q, lam, c0, g, ap.b, faci, faciq); break;
    case 1: load_neighbours<NB, NQ, 0, 1>(kn, q, lam, c0, g, ap.b, faci, faciq); break;
    case 2: load_neighbours<NB, NQ, 1, 0>(kn, q, lam, c0, g, ap.b, faci, faciq); break;
    case 3: load_neighbours<NB, NQ, 1, 1>(kn, q, lam, c0, g, ap.b, faci, faciq); break;
    case 4: load_neighbours<NB, NQ, 2, 0>(kn, q, lam, c0, g, ap.b, faci, faciq); break;
    case 5: load_neighbours<NB, NQ, 2, 1>(kn, q, lam, c0, g, ap.b, faci, faciq); break;
    }
    __syncthreads();
    switch (wave) {
    case 0: face_point_vjp<NB, QP, NQ, RM, 0, 0>(kn, m_s, lo_s, c0, g, ph, ap.inflow); break;
    case 1: face_point_vjp<NB, QP, NQ, RM, 0, 1>(kn, m_s, lo_s, c0, g, ph, ap.inflow); break;
    case 2: face_point_vjp<NB, QP, NQ, RM, 1, 0>(kn, m_s, lo_s, c0, g, ph, ap.inflow); break;
    case 3: face_point_vjp<NB, QP, NQ, RM, 1, 1>(kn, m_s, lo_s, c0, g, ph, ap.inflow); break;
    case 4: face_point_vjp<NB, QP, NQ, RM, 2, 0>(kn, m_s, lo_s, c0, g, ph, ap.inflow); break;
    case 5: face_point_vjp<NB, QP, NQ, RM, 2, 1>(kn, m_s, lo_s, c0, g, ph, ap.inflow); break;
    default: {
        const int v = t - 384, p = v / C, c = v % C;
        double bQ[NQ];
        volume_point_vjp<NB, NQ>(m_s + c * NB, lo_s + c * NB, C * NB, T->bint[p], 0.25 * T->w3[p], g, ph, bQ);
#pragma unroll
        for (int f = 0; f < NQ; f++) bq_s[f][v] = bQ[f];
        if (ap.q_raw && v >= 64 && v < 64 + C)
            limit_terms<NB, QP>(ap, g, c0 + c < g.N ? c0 + c : g.N - 1, lim_s[c], th_s[0][c], th_s[1][c]);
    }
    }
    __syncthreads();
    double dcoll = 0.;
    for (int it = t; it < NQ * C; it += 512) {
        const int f = it / C, lc = it % C;
        const long c = c0 + lc;
        if (c >= g.N) continue;
        double rt[NB];
#pragma unroll
        for (int r = 0; r < NB; r++) rt[r] = 0.;
#pragma unroll
        for (int p = 0; p < NPG; p++) {
            const double v = bq_s[f][p * C + lc];
#pragma unroll
            for (int r = 0; r < NB; r++) rt[r] += fz::phi_int<NB, QP>(r, p / (QP * QP), (p / QP) % QP, p % QP) * v;
        }
#pragma unroll
        for (int w = 0; w < 6; w++)
#pragma unroll
            for (int p = 0; p < NF; p++) {
                const double v = kn_s[w][f * 64 + p * C + lc];
#pragma unroll
                for (int r = 0; r < NB; r++) rt[r] += fz::phi_face<NB, QP>(w / 2, w % 2, r, p / QP, p % QP) * v;
            }
        dcoll += field_finish<NB, NQ>(lam, lam_in, g, ap, f, c, dt, faci, m_s + (f * C + lc) * NB, lo_s + lc * NB,
                                      C * NB, lim_s[lc], th_s[0][lc], th_s[1][lc], rt);
    }
    if (ap.partial) block_partial_of<8>(dcoll, ap.partial);
}

// ------------------------------------------------- 13-moment transpose ----
// The transpose of a 13-moment stage on a grid periodic in every direction,
// split into a face and a cell kernel, so that no lane holds a whole cell.
// Both take a workgroup's quadrature points side by side, one point of one
// face or cell a lane: the modes wait in LDS, where each lane reads what its
// point needs, and the points' cotangents go back through LDS to be summed.
// The face kernel writes, for each side of a face, the moments
// M_k = sum_p b_k(p) v(p) of the cotangents v of that side's trace (NK values
// a field instead of QP^2); the cell kernel adds the volume transpose and
// gathers its six faces.  The sum over the terms is k_stage_vjp's, evaluated
// in another order.  A periodic grid has as many faces a direction as cells:
// face c is the low face of cell c.
// nbasis 10, Roe, 40^3 cells, a stage: 217 us the faces (three directions in
// one launch, 51 KB of LDS: three workgroups a CU) and 201 us the cells,
// against 840 and 429 us for a wave per face point over 64 faces (156 KB of
// LDS, one workgroup a CU, waiting for its loads two thirds of the time, and
// a last round of one workgroup) and a field per wave (three of thirteen
// waves at the points).  Bound by the arithmetic of the points at three or
// four waves a SIMD, then by L2: 0.6 GB a stage.

// Faces of a workgroup of 256: as many as give every lane a face point.
template <int QP>
constexpr int face13_faces() { return 256 / (QP * QP); }
template <int NB, int QP>
constexpr int face13_doubles() {
    const int modes = 3 * 13 * fz::face_nk<NB>() * face13_faces<QP>(), points = 2 * 13 * QP * QP * face13_faces<QP>();
    return modes > points ? modes : points;
}

// The faces f0.. of direction DIR: each field's trace coefficients of both
// sides and the sum of their lifted-cotangent coefficients (of b*lam through
// the relaxation factors) to LDS; then at each point the cotangent mu of the
// flux, reversed through the Riemann solver and the physical fluxes; then the
// moments of both sides' trace cotangents.
template <int NB, int QP, int RM, int DIR>
__device__ __forceinline__ void face13_vjp(double* __restrict__ lds, const double* __restrict__ q,
                                           const double* __restrict__ lam, double* __restrict__ ml,
                                           double* __restrict__ mr, long f0, const Grid& g, const Phys& ph,
                                           const AdjParams& ap) {
    constexpr int NQ = 13, NF = QP * QP, NK = fz::face_nk<NB>(), F = face13_faces<QP>();
    const double dt = *ap.dt;
    const double faci = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll) : 1.0;
    const double faciq = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll_q) : 1.0;
    const auto& FP = fz::face_poly<NB>();
    const int t = (int)threadIdx.x;
    for (int it = t; it < NQ * F; it += 256) {
        const int l = it % F, fld = it / F;
        const long cr = f0 + l < g.N ? f0 + l : g.N - 1;
        const long sd = DIR == 0 ? 1 : DIR == 1 ? g.nx : (long)g.nx * g.ny;
        const int n_ax = DIR == 0 ? g.nx : DIR == 1 ? g.ny : g.nz;
        const int a = (int)(DIR == 0 ? cr % g.nx : DIR == 1 ? (cr / g.nx) % g.ny : cr / ((long)g.nx * g.ny));
        const long cl = a == 0 ? cr + (n_ax - 1) * sd : cr - sd;
        const double fac = ap.b * (fld >= T_QX ? faciq : (fld >= PXX ? faci : 1.0));
        double m0[1][NB], m1[1][NB], l0[1][NB], l1[1][NB], K0[1][NK], K1[1][NK], L0[1][NK], L1[1][NK];
#pragma unroll
        for (int r = 0; r < NB; r++) {
            const long o = ((long)r * NQ + fld) * g.N;
            m0[0][r] = q[o + cl];
            m1[0][r] = q[o + cr];
            l0[0][r] = lam[o + cl];
            l1[0][r] = lam[o + cr];
        }
        sg::signed_coeffs<NB, 1, DIR, NK>(m0, 1.0, K0);
        sg::signed_coeffs<NB, 1, DIR, NK>(m1, -1.0, K1);
        lift_coeffs<NB, 1, DIR, 1, NK>(l0, L0);
        lift_coeffs<NB, 1, DIR, 0, NK>(l1, L1);
        double* const k = lds + it * NK;
#pragma unroll
        for (int e = 0; e < NK; e++) {
            k[e] = K0[0][e];
            k[NQ * F * NK + e] = K1[0][e];
            k[2 * NQ * F * NK + e] = fac * (L0[0][e] + L1[0][e]);
        }
    }
    __syncthreads();
    const bool point = t < NF * F;
    double bL[NQ], bR[NQ];
    if (point) {
        const int p = t / F, l = t % F;
        const double dxi_d = DIR == 0 ? g.dxi : DIR == 1 ? g.dyi : g.dzi;
        double b[NK], wb[NK];
#pragma unroll
        for (int e = 0; e < NK; e++) {
            b[e] = FP.b[p][e];
            wb[e] = dxi_d * FP.wb[p][e];
        }
        // field f of a side's state (by the forward kernel's functions, so that
        // every Riemann branch is taken as in the forward stage), or (side 2,
        // with wb) of the flux's cotangent
        auto value = [&](int side, int f, const double (&w)[NK]) {
            const double* const k = lds + ((side * NQ + f) * F + l) * NK;
            if (side < 2) return sg::eval_one<NK>(k, w);
            double s = k[0] * w[0];
#pragma unroll
            for (int e = 1; e < NK; e++) s += k[e] * w[e];
            return s;
        };
        // face_vjp in three parts (the Riemann solver's Euler fields, the
        // left flux, the right flux), so that no part holds all that the
        // point has: 13 fields of two states and of their cotangents at once
        // spilled 480 registers
        double QL[NQ], QR[NQ], mu[NQ], bFL[NQ], bFR[NQ];
#pragma unroll
        for (int f = 0; f < NQ; f++) {
            bL[f] = 0.;
            bR[f] = 0.;
        }
#pragma unroll
        for (int f = 0; f < 5; f++) {
            QL[f] = value(0, f, b);
            QR[f] = value(1, f, b);
            mu[f] = value(2, f, wb);
        }
        riemann_vjp<RM, DIR>(ph, QL, QR, mu, bL, bR, bFL, bFR);
        sg::section();
#pragma unroll
        for (int f = 5; f < NQ; f++) {
            QL[f] = value(0, f, b);
            bFL[f] = 0.5 * value(2, f, wb);
        }
        flux_vjp<NQ, DIR>(ph, QL, pr::prim<NQ>(ph, QL), bFL, bL);
        sg::section();
#pragma unroll
        for (int f = 5; f < NQ; f++) {
            QR[f] = value(1, f, b);
            bFR[f] = 0.5 * value(2, f, wb);
        }
        flux_vjp<NQ, DIR>(ph, QR, pr::prim<NQ>(ph, QR), bFR, bR);
    }
    __syncthreads();  // the points' cotangents overwrite the coefficients
    if (point) {
#pragma unroll
        for (int f = 0; f < NQ; f++) {
            lds[f * NF * F + t] = bL[f];
            lds[(NQ + f) * NF * F + t] = bR[f];
        }
    }
    __syncthreads();
    for (int it = t; it < 2 * NQ * F; it += 256) {
        const int l = it % F, row = it / F;  // row: side, field
        double M[NK];
#pragma unroll
        for (int p = 0; p < NF; p++) {
            const double v = lds[(row * NF + p) * F + l];
#pragma unroll
            for (int e = 0; e < NK; e++) M[e] = p == 0 ? v * FP.b[p][e] : M[e] + v * FP.b[p][e];
        }
        if (f0 + l < g.N) {
            double* const out = row < NQ ? ml + (long)row * NK * g.N : mr + (long)(row - NQ) * NK * g.N;
#pragma unroll
            for (int e = 0; e < NK; e++) out[e * g.N + f0 + l] = M[e];
        }
    }
}

// All three directions in one launch, a tile's directions next to each other
// and each XCD a contiguous eighth of the tiles (L2 serves the cells that
// several faces share).
template <int NB, int QP, int RM>
__global__ __launch_bounds__(256, (NB == 10 ? 3 : 2)) void k_face13_vjp(
    const double* __restrict__ q, const double* __restrict__ lam, double* __restrict__ ml0,
    double* __restrict__ ml1, double* __restrict__ ml2, double* __restrict__ mr0, double* __restrict__ mr1,
    double* __restrict__ mr2, Grid g, Phys ph, AdjParams ap) {
    __shared__ __attribute__((aligned(16))) double lds[face13_doubles<NB, QP>()];
    const unsigned b = xcd_block();  // the grid is a multiple of 8
    const unsigned tile = b / 3, d = b % 3;
    const long f0 = (long)tile * face13_faces<QP>();
    if (f0 >= g.N) return;
    if (d == 0) face13_vjp<NB, QP, RM, 0>(lds, q, lam, ml0, mr0, f0, g, ph, ap);
    else if (d == 1) face13_vjp<NB, QP, RM, 1>(lds, q, lam, ml1, mr1, f0, g, ph, ap);
    else face13_vjp<NB, QP, RM, 2>(lds, q, lam, ml2, mr2, f0, g, ph, ap);
}

// Cells of a workgroup of k_cell13_vjp, and its lanes: a volume point each,
// and one more wave for the limiter's factors.
template <int QP>
constexpr int cell13_cells() { return QP == 3 ? 16 : 32; }
template <int QP>
constexpr int cell13_threads() { return (QP * QP * QP * cell13_cells<QP>() + 63) / 64 * 64 + 64; }

// The cells' modes and cotangents to LDS; then a volume point a lane: its
// state, the cotangents of its three fluxes (the transposes of the volume
// sums), the fluxes reversed (flux_vjp) and the state cotangent to LDS; then
// a field of a cell a lane: the points' sum, the face moments (the cell is
// the right side of its low faces and the left side of its high faces), the
// sources, the stage map (lo + dt*rt, the accumulated terms) and the frozen
// limiter, as cell_vjp_finish; d/dcoll as cell_vjp_parts.
template <int NB, int QP, int RM>
__global__ __launch_bounds__(cell13_threads<QP>(), 4) void k_cell13_vjp(
    const double* __restrict__ q, const double* __restrict__ lam, double* __restrict__ lam_in,
    const double* __restrict__ ml0, const double* __restrict__ ml1, const double* __restrict__ ml2,
    const double* __restrict__ mr0, const double* __restrict__ mr1, const double* __restrict__ mr2,
    const Tables* __restrict__ T, Grid g, Phys ph, AdjParams ap) {
    constexpr int NQ = 13, NPG = QP * QP * QP, NK = fz::face_nk<NB>(), C = cell13_cells<QP>();
    constexpr int NT = cell13_threads<QP>();
    __shared__ __attribute__((aligned(16))) double m_s[NQ][C][NB], lo_s[NQ][C][NB];
    __shared__ double bq_s[NQ][NPG * C];
    __shared__ double th_s[2][C];
    __shared__ int lim_s[C];
    const int t = (int)threadIdx.x;
    const long c0 = (long)xcd_block() * C;
    const double dt = *ap.dt;
    const double faci = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll) : 1.0;
    const double faciq = (ap.ivis == 1 && !ap.rhs_only) ? 1. / (1. + dt * ap.coll_q) : 1.0;
#pragma unroll
    for (int n = 0; n < (NQ * NB * C + NT - 1) / NT; n++) {
        const int it = t + n * NT;
        if (it < NQ * NB * C) {
            const int c = it % C, row = it / C, r = row / NQ, f = row % NQ;
            // lanes past the grid take a copy of the last cell and store nothing
            const long o = (long)row * g.N + (c0 + c < g.N ? c0 + c : g.N - 1);
            m_s[f][c][r] = q[o];
            lo_s[f][c][r] = ap.b * lam[o] * (f >= T_QX ? faciq : (f >= PXX ? faci : 1.0));
        }
    }
    __syncthreads();
    if (t < NPG * C) {
        const int p = t / C, c = t % C;
        double bQ[NQ];
        volume_point_vjp<NB, NQ>(&m_s[0][c][0], &lo_s[0][c][0], C * NB, T->bint[p], 0.25 * T->w3[p], g, ph, bQ);
#pragma unroll
        for (int f = 0; f < NQ; f++) bq_s[f][t] = bQ[f];
    } else if (ap.q_raw && t >= NT - 64 && t < NT - 64 + C) {
        const int c = t - (NT - 64);
        const long cc = c0 + c < g.N ? c0 + c : g.N - 1;
        limit_terms<NB, QP>(ap, g, cc, lim_s[c], th_s[0][c], th_s[1][c]);
    }
    __syncthreads();
    double dcoll = 0.;
    for (int it = t; it < NQ * C; it += NT) {
        const int f = it / C, lc = it % C;
        const long c = c0 + lc;
        if (c >= g.N) continue;
        double rt[NB];
#pragma unroll
        for (int r = 0; r < NB; r++) rt[r] = 0.;
#pragma unroll
        for (int p = 0; p < NPG; p++) {
            const double v = bq_s[f][p * C + lc];
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const double b = fz::phi_int<NB, QP>(r, p / (QP * QP), (p / QP) % QP, p % QP);
                if (b != 0.) rt[r] += b * v;
            }
        }
        const int i = (int)(c % g.nx), j = (int)((c / g.nx) % g.ny), k = (int)(c / ((long)g.nx * g.ny));
        const long nxy = (long)g.nx * g.ny;
        const long ch[3] = {i == g.nx - 1 ? c - i : c + 1, j == g.ny - 1 ? c - (long)j * g.nx : c + g.nx,
                            k == g.nz - 1 ? c - k * nxy : c + nxy};
        const double* const ml[3] = {ml0, ml1, ml2};
        const double* const mr[3] = {mr0, mr1, mr2};
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double ML[NK], MR[NK];
#pragma unroll
            for (int e = 0; e < NK; e++) {
                MR[e] = mr[d][((long)f * NK + e) * g.N + c];
                ML[e] = ml[d][((long)f * NK + e) * g.N + ch[d]];
            }
#pragma unroll
            for (int r = 0; r < NB; r++) {
                const int e = fz::pair_index(fz::deg<NB>(r, fz::row_axis(d)), fz::deg<NB>(r, fz::col_axis(d)));
                rt[r] += fz::Lface(fz::deg<NB>(r, d), 0) * MR[e] + ML[e];
            }
        }
        dcoll += field_finish<NB, NQ>(lam, lam_in, g, ap, f, c, dt, faci, &m_s[f][lc][0], &lo_s[0][lc][0], C * NB,
                                      lim_s[lc], th_s[0][lc], th_s[1][lc], rt);
    }
    if (ap.partial) block_partial_of<NT / 64>(dcoll, ap.partial);
}

// adds the block partials to *acc (one block, fixed order)
static __global__ __launch_bounds__(256) void k_sum_partials(const double* __restrict__ partial, int n,
                                                             double* __restrict__ acc) {
    __shared__ double red[4];
    double s = 0.;
    for (int b = threadIdx.x; b < n; b += blockDim.x) s += partial[b];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += red[w];
        *acc += t;
    }
}

}  // namespace adj
}  // namespace hd
