// hd_prim.h -- point physics written around shared primitive variables, for
// the fused kernels: each state's 1/rho, velocity and pressures are computed
// once and used by both the physical flux (flux_calc_pnts_r,
// src/flux.f90:23-193) and the Riemann solver (flux_hllc, src/flux.f90:466-647),
// which in the reference recompute them separately.  Reciprocals use the
// hardware estimate refined by two Newton steps (faithful in FP64), which
// agrees with IEEE division to an ulp; the reference's formulas are otherwise
// kept term by term.
#pragma once
#include "hd_physics.h"

namespace hd {
namespace pr {

__device__ __forceinline__ double rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    r = fma(fma(-x, r, 1.0), r, r);
    return r;
}
// a/b with one residual correction on top of the refined reciprocal
__device__ __forceinline__ double divide(double a, double b) {
    const double r = rcp(b);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

struct Prim {
    double ri;       // 1/rho
    double u[3];     // velocity
    double pf;       // flux pressure: max(gm1*(E - 0.5/rho*|m|^2), P_floor)
};

template <int NQ>
__device__ __forceinline__ Prim prim(const Phys& ph, const double* Q) {
    Prim s;
    s.ri = rcp(Q[RH]);
    s.u[0] = Q[MX] * s.ri;
    s.u[1] = Q[MY] * s.ri;
    s.u[2] = Q[MZ] * s.ri;
    const double smsq = Q[MX] * Q[MX] + Q[MY] * Q[MY] + Q[MZ] * Q[MZ];
    double P = ph.gm1 * (Q[EN] - 0.5 * s.ri * smsq);
    s.pf = P < ph.P_floor ? ph.P_floor : P;
    return s;
}

// Numerator of the HLLC contact speed, aR*uR - aL*uL + pL - pR, rounded
// product by product: at a mirror state (the x-high outflow ghost reverses
// the normal momentum) it is exactly zero, and a fused multiply-add would
// leave a signed rounding residue that picks a different star state than
// the reference's arithmetic does.
__device__ __forceinline__ double contact_num(double aR, double uR, double aL, double uL, double pL, double pR) {
#pragma clang fp contract(off)
    return aR * uR - aL * uL + pL - pR;
}

// sqrt by the hardware estimate of 1/sqrt and two Goldschmidt steps, accurate
// to an ulp; 0 for 0, NaN below 0.
__device__ __forceinline__ double root(double x) {
    double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    return x == 0.0 ? x : g;
}

// 1/rho, the velocity and the pressure (no floor) of one side of a face.  Shared
// with the transpose, and rounded operation by operation, so that both see the
// same values whatever the compiler makes of the code around them.
struct Side {
    double ri, u[3], p;
};
__device__ __forceinline__ Side side(const Phys& ph, const double* Q) {
#pragma clang fp contract(off)
    Side s;
    s.ri = rcp(Q[RH]);
#pragma unroll
    for (int a = 0; a < 3; a++) s.u[a] = Q[MX + a] * s.ri;
    s.p = ph.gm1 * fma(-0.5, fma(Q[MX], s.u[0], fma(Q[MY], s.u[1], Q[MZ] * s.u[2])), Q[EN]);
    return s;
}

// HLLC's speeds and the branch they select (Batten 1997 with Davis speeds, the
// order of the branches hllc_point's): the last true of SL > 0 (left), SL <= 0 <
// SM (left star), SM <= 0 <= SR (right star), SR < 0 (right); none of them with
// NaN speeds.  One function for the flux and its transpose: at rest the contact
// speed is a difference of equal pressures, and with stress the flux jumps where
// it changes sign.
struct HllcSpeeds {
    double cL, cR, SL, SR, SM, aL, aR, den;  // SM = contact_num / den
    bool den_floor;
    int sel;  // 0 left, 1 left star, 2 right star, 3 right, -1 none
};
template <int DIR>
__device__ __forceinline__ HllcSpeeds hllc_speeds(const Phys& ph, double rL, const Side& L, double rR, const Side& R) {
#pragma clang fp contract(off)
    HllcSpeeds w;
    const double nL = L.u[DIR], nR = R.u[DIR];
    w.cL = root(ph.gamma * L.p * L.ri);
    w.cR = root(ph.gamma * R.p * R.ri);
    w.SL = fmin(nL - w.cL, nR - w.cR);
    w.SR = fmax(nR + w.cR, nL + w.cL);
    w.aR = rR * (w.SR - nR);
    w.aL = rL * (w.SL - nL);
    w.den = w.aR - w.aL;
    w.den_floor = w.den == 0.0;
    if (w.den_floor) w.den = ph.rh_floor;
    w.SM = divide(contact_num(w.aR, nR, w.aL, nL, L.p, R.p), w.den);
    w.sel = -1;
    if (w.SL > 0.0) w.sel = 0;
    if (w.SL <= 0.0 && 0.0 < w.SM) w.sel = 1;
    if (w.SM <= 0.0 && 0.0 <= w.SR) w.sel = 2;
    if (w.SR < 0.0) w.sel = 3;
    return w;
}

// Roe flux (roe_point: Eulderink and Mellema, half the thermal enthalpy) from
// the traces' velocities, pressures and 1/rho, with refined reciprocals and
// roots; out holds 0.5 (FL + FR) on entry.
template <int DIR>
__device__ __forceinline__ void roe_diss(const Phys& ph, const double* QL, const double* QR, double riL, double riR,
                                         const double* uL, const double* uR, double pL, double pR, double* out) {
    constexpr int IP = MX + DIR, I1 = MX + (DIR + 1) % 3, I2 = MX + (DIR + 2) % 3;
    constexpr int A = DIR, B = (DIR + 1) % 3, C = (DIR + 2) % 3;
    const double cp = ph.gamma * ph.gm1i;
    const double kL = root(QL[RH]), kR = root(QR[RH]), ki = rcp(kL + kR);
    const double hL = fma(uL[0], uL[0], fma(uL[1], uL[1], fma(uL[2], uL[2], cp * (pL * riL))));
    const double hR = fma(uR[0], uR[0], fma(uR[1], uR[1], fma(uR[2], uR[2], cp * (pR * riR))));
    const double v0 = fma(kL, uL[A], kR * uR[A]) * ki, v1 = fma(kL, uL[B], kR * uR[B]) * ki,
                 v2 = fma(kL, uL[C], kR * uR[C]) * ki, h = 0.5 * (fma(kL, hL, kR * hR) * ki);
    const double hv = 0.5 * fma(v0, v0, fma(v1, v1, v2 * v2));
    const double asq = ph.gm1 * (h - hv);
    if (__builtin_expect(!(asq > 0.0), 0)) {
        // no Roe sound speed: local Lax-Friedrichs, as the legacy code
        const double cw = fmax(fabs(uL[A]) + root(ph.gamma * pL * riL), fabs(uR[A]) + root(ph.gamma * pR * riR));
#pragma unroll
        for (int f = 0; f < 5; f++) out[f] -= 0.5 * cw * (QR[f] - QL[f]);
        return;
    }
    const double ai = rcp(asq), a = root(asq);
    const double dr = fma(QR[RH], riL, -1.), de = (QR[EN] - QL[EN]) * riL, dn = (QR[IP] - QL[IP]) * riL,
                 d1 = (QR[I1] - QL[I1]) * riL, d2 = (QR[I2] - QL[I2]) * riL;
    const double ea = ph.gm1 * ai;
    const double vd = fma(v0, dn, fma(v1, d1, fma(v2, d2, -de)));
    const double ev = 0.5 * ea * fma(hv, dr, -vd), od = 0.5 * fma(-v0, dr, dn) * (a * ai);
    const double l2 = fabs(v0);
    const double t0 = (ev - od) * fabs(v0 - a), t1 = (ev + od) * fabs(v0 + a);
    const double t2 = ea * fma(h - 2. * hv, dr, vd) * l2, t3 = fma(-v1, dr, d1) * l2, t4 = fma(-v2, dr, d2) * l2;
    const double sr = t0 + t1 + t2, hl = -0.5 * QL[RH];
    out[RH] = fma(hl, sr, out[RH]);
    out[IP] = fma(hl, fma(v0, sr, a * (t1 - t0)), out[IP]);
    out[I1] = fma(hl, fma(v1, sr, t3), out[I1]);
    out[I2] = fma(hl, fma(v2, sr, t4), out[I2]);
    out[EN] = fma(hl, fma(h, t0 + t1, fma(a * v0, t1 - t0, fma(hv, t2, fma(v1, t3, v2 * t4)))), out[EN]);
}

// Flux through one face point from the two traces: rh..en by the Riemann
// solver RM, and with stress (NQ >= 11, traces holding rh..en and row DIR of
// the stress) the averaged velocity in F[5..7], to which the central fluxes
// of the stress rows are proportional; with 13 moments (traces holding also
// the heat flux along DIR) the averaged temperature in F[8].  S: the row of
// the stochastic stress.
// HLLC keeps density, velocity and pressure of both sides, selects one, and
// forms the conserved values and the flux of that side only (few values are
// live at a time; the momentum and energy come back to rounding).
template <int NQ, int DIR, int RM, bool NZ>
__device__ __forceinline__ void face_flux(const Phys& ph, const double* QL, const double* QR, const double* S,
                                          double* F) {
    constexpr int IP = MX + DIR;
    const double rL = QL[RH], rR = QR[RH];
    const Side L = side(ph, QL), R = side(ph, QR);
    const double riL = L.ri, riR = R.ri, pL = L.p, pR = R.p;
    const double (&uL)[3] = L.u, (&uR)[3] = R.u;
    if constexpr (NQ >= 11) {
#pragma unroll
        for (int a = 0; a < 3; a++) F[5 + a] = 0.5 * (uL[a] + uR[a]);
    }
    if constexpr (NQ == 13)
        F[8] = 0.5 * ((pL < ph.P_floor ? ph.P_floor : pL) * riL + (pR < ph.P_floor ? ph.P_floor : pR) * riR);
    // physical flux of one side: floored pressure, stress row less the noise
    auto side_flux = [&](const double* Q, const double* u, double p, const double* P3, double* f) {
        const double pf = p < ph.P_floor ? ph.P_floor : p;
        const double un = u[DIR];
        f[RH] = Q[IP];
        f[EN] = (Q[EN] + pf) * un;
        if constexpr (NQ >= 11) {
            double Pn[3];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                Pn[a] = P3[a];
                if constexpr (NZ) Pn[a] -= S[a];
                f[MX + a] = fma(Q[MX + a], un, a == DIR ? Pn[a] + pf : Pn[a]);
            }
            f[EN] += fma(Pn[0], u[0], fma(Pn[1], u[1], Pn[2] * u[2]));
            if constexpr (NQ == 13) f[EN] += P3[3];
        } else {
#pragma unroll
            for (int a = 0; a < 3; a++) f[MX + a] = a == DIR ? fma(Q[MX + a], un, pf) : Q[MX + a] * un;
        }
    };
    if constexpr (RM != RIEMANN_HLLC) {
        double FL[5], FR[5];
        side_flux(QL, uL, pL, QL + 5, FL);
        side_flux(QR, uR, pR, QR + 5, FR);
#pragma unroll
        for (int f = 0; f < 5; f++) F[f] = 0.5 * (FL[f] + FR[f]);
        if constexpr (RM == RIEMANN_ROE) roe_diss<DIR>(ph, QL, QR, riL, riR, uL, uR, pL, pR, F);
        return;
    }
    const HllcSpeeds w = hllc_speeds<DIR>(ph, rL, L, rR, R);
    const double SL = w.SL, SR = w.SR, SM = w.SM;
    const double pstar = fma(-w.aL, uL[DIR] - SM, pL);  // Eq. (36)
    // NaN speeds: the central flux (the reference's default), before the
    // selection so that only one side's values are live after it
    const bool none = w.sel < 0;
    if (__builtin_expect(none, 0)) {
        double FL[5], FR[5];
        side_flux(QL, uL, pL, QL + 5, FL);
        side_flux(QR, uR, pR, QR + 5, FR);
#pragma unroll
        for (int e = 0; e < 5; e++) F[e] = 0.5 * (FL[e] + FR[e]);
    }
    const bool right = w.sel >= 2;
    const double r = right ? rR : rL, p = right ? pR : pL, Sk = right ? SR : SL;
    double u[3], P3[4] = {0., 0., 0., 0.}, Q[5], f[5];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        u[a] = right ? uR[a] : uL[a];
        if constexpr (NQ >= 11) P3[a] = right ? QR[5 + a] : QL[5 + a];
    }
    if constexpr (NQ == 13) P3[3] = right ? QR[8] : QL[8];
    if (none) return;
    Q[RH] = r;
#pragma unroll
    for (int a = 0; a < 3; a++) Q[MX + a] = r * u[a];
    Q[EN] = fma(0.5, fma(Q[MX], u[0], fma(Q[MY], u[1], Q[MZ] * u[2])), p * ph.gm1i);
    side_flux(Q, u, p, P3, f);
    if (w.sel == 0 || w.sel == 3) {  // supersonic: the side's own flux
#pragma unroll
        for (int e = 0; e < 5; e++) F[e] = f[e];
        return;
    }
    double den = Sk - SM;
    if (den == 0.0) den = ph.rh_floor;
    const double sr = Sk * rcp(den);
    // F + Sk*(Q* - Q) with Q* = (Sk - un)/(Sk - SM) Q + pressure terms
    const double ga = fma(sr, Sk - u[DIR], -Sk);
#pragma unroll
    for (int e = 0; e < 5; e++) F[e] = fma(ga, Q[e], f[e]);
    F[IP] = fma(sr, pstar - p, F[IP]);
    F[EN] = fma(sr, fma(pstar, SM, -(p * u[DIR])), F[EN]);
}

}  // namespace pr
}  // namespace hd
