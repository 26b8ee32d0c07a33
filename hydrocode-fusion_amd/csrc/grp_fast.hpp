// grp_fast.hpp -- the interface solver of the time steps in the arithmetic of
// fast_arith.hpp: the same results, bit for bit, as riemann_exact, grp_q1d and
// grp_2d_flux* (grp_device.hpp) give with IEEE division and square root, for
// sides whose values are far from the ends of the exponent range.
//
// What bounds the steps is the number of FP64 instructions of one interface
// (the sweeps issue VALU instructions 55-75 % of the time), and half of them
// were division and square root expansions.  Here a divisor's reciprocal is
// formed once (the states' own, the wave's root) and each quotient by it takes
// 3 instructions instead of 11; the root and its reciprocal of the wave curve
// are kept for the Newton slope at the same pressure, which took them again;
// terms that the split path multiplies by its zero tangential derivatives are
// not there; the update by the wave the t-axis lies in is written once for
// both sides.  What is left out can only change the sign of a zero.
//
// sides_in_range says which interfaces may come here; the solver itself gives
// up (returns false) where the star pressure leaves the range.  The steps then
// solve that face again with the IEEE solver, out of line and from its cells in
// memory, so that nothing is kept in registers for it.
#pragma once
#include "fast_arith.hpp"
#include "grp_device.hpp"

namespace hgrp {

// ---- which interfaces -------------------------------------------------------------
HGRP_HD bool tiny(double x) { return fabs(x) < 0x1p-300 && x != 0.0; }

// Densities and pressures in [LEAST, MOST], velocities and derivatives below
// MOST; derivatives of density and pressure zero or differences of such values
// over h.  7e-40 to 1e39 holds gas in the usual units: an interface that is left
// to the IEEE solver costs more than it did before there were two (512^2 with the
// learned guess, left there .397 ms a step, taken here .156, .260 by the IEEE
// solver alone).
// Ahead of a front velocities decay cell by cell through every magnitude down to
// the denormals, over regions tens of cells wide, while differences of pressure
// and density stop at their rounding: so what may be a velocity (or a fraction)
// by itself is divided by IEEE division in the acoustic case and in the passive
// members, and after the Riemann solve where a wave holds such an interface
// (div_r).
HGRP_HD double magnitude(const Side &S)           // of the velocities and derivatives; NaN for a NaN
{
    return ((fabs(S.u) + fabs(S.v)) + (fabs(S.d_rho) + fabs(S.d_u))) + (fabs(S.d_v) + fabs(S.d_p));
}
static constexpr double LEAST = 0x1p-130, MOST = 0x1p130;
HGRP_HD bool sides_in_range(const Side &L, const Side &R)
{
    return L.rho >= LEAST && L.p >= LEAST && R.rho >= LEAST && R.p >= LEAST &&
           fmax(fmax(L.rho, L.p), fmax(R.rho, R.p)) <= MOST && magnitude(L) + magnitude(R) <= MOST;
}
// a / rho, b / rho, c / rho of a cell's update
__device__ __forceinline__ void quot3(double a, double b, double c, double rho, double &qa, double &qb, double &qc)
{
    const Rcp r = rcp_of(rho);
    qa = div_q(a, r);
    qb = div_q(b, r);
    qc = div_q(c, r);
    const bool in = rho >= LEAST && rho <= MOST && fmax(fmax(fabs(a), fabs(b)), fabs(c)) <= 0x1p300 &&
                    !tiny(c);
    if (tiny(a) || tiny(b)) {                    // a momentum ahead of a front
        qa = a / rho;
        qb = b / rho;
    }
    if (__builtin_expect(!in, 0)) {
        const Quot4 q = quot4_slow(a, b, c, 0.0, rho);
        qa = q.q[0];
        qb = q.q[1];
        qc = q.q[2];
    }
}
HGRP_HD bool any_lane(bool x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __any(x);
#else
    return x;
#endif
}
// a / r.b; rough (the same for the whole wave): a may be tiny
HGRP_HD double div_r(double a, const Rcp &r, bool rough) { return rough ? a / r.b : div_q(a, r); }

HGRP_HD bool gas_in_range(const Gas &G) { return G.gm1() >= 0x1p-20 && G.g <= 0x1p20; }

// ---- the exact Riemann solve ---------------------------------------------------------
// What the wave curve leaves for the Newton slope at the same pressure and, from
// the last one, for the state behind the wave: on the rarefaction branch
// l = log(p/p_s) and m = (p/p_s)^mu; on the shock branch m = 0 and l is
// sqrt(1 + nu (p - p_s)/p_s) with its reciprocal (an Rcp).
struct Keep {
    DD l;
    double m;
};
template <int SIGN>
HGRP_HD double curve_q(double p, double u_s, const Rcp &p_s, double c_s, const Gas &G, Keep *keep, const double *P)
{
    double w;
    if (p > p_s.b) {
        const double dp = p - p_s.b;
        const Rcp s = rcp_of(sqrt_q(1.0 + div_q(G.nu * dp, p_s)));
        keep->l = {s.b, s.y};
        keep->m = 0.0;
        w = div_q(div_q(div_q(dp * c_s, {G.g, G.inv_g}), p_s), s);
    } else {
        keep->l = log_in_range(div_q(p, p_s), P);
        keep->m = pow_in_range(keep->l, G.mu, P);
        w = keep->m - 1.0;
        w = div_q(2.0 * c_s * w, {G.gm1(), G.y_gm1});
    }
    return SIGN < 0 ? u_s - w : u_s + w;
}

// dv/dp along the 3-wave (the 1-wave's is its negative) at the pressure of the last curve_q
HGRP_HD double slope_q(double p, const Rcp &p_s, double c_s, const Gas &G, const Keep &keep, const double *P)
{
    const double t2 = div_q(div_q(c_s, {G.g, G.inv_g}), p_s);
    if (p > p_s.b) {
        const double t1 = recip_q({keep.l.hi, keep.l.lo});
        const double t3 = div_q(0.5 * t2 * G.nu, p_s);
        return t2 * t1 - t3 * (p - p_s.b) * cube(t1);
    }
    return recip_1(pow_in_range(keep.l, G.nu, P)) * t2;
}

struct StarQ {
    double u, p;
    int crw0, crw1;
};

// The iteration: the star pressure p, the curves' velocities v_L and v_R at it,
// the star velocity u.
template <bool CONV, int N>
HGRP_HD bool newton_q(const Gas &GL, const Gas &GR, double u_L, double u_R, const Rcp &p_L, const Rcp &p_R, double c_L,
                      double c_R, double tol, double p_guess, double &p, double &v_L, double &v_R, double &u, Keep &kL,
                      Keep &kR, const double *P)
{
    // the states of riemann_exact's loop: 0 the curves at the learned guess, 1 steps from it,
    // 2 the curves at the reference's guess, 3 steps from it, 4 and 5 the converge rule's extra steps
    int st = p_guess > 0.0 ? 0 : 2, n = 0, done = 0;
    double k1 = 0.0, k3 = 0.0;
    p = p_guess;
    for (;;) {
        if (st == 0 || st == 2) {
            k1 = div_q(div_q(-c_L, p_L), {GL.g, GL.inv_g});
            k3 = div_q(div_q(c_R, p_R), {GR.g, GR.inv_g});
            if (st == 2) {
                double p0 = div_1(k1 * p_L.b - k3 * p_R.b - u_L + u_R, k1 - k3);
                if (p0 < 0) p0 = (p_L.b < p_R.b) ? p_L.b : p_R.b;
                p = 0.5 * p0;
            }
        } else {
            k1 = -slope_q(p, p_L, c_L, GL, kL, P);
            k3 = slope_q(p, p_R, c_R, GR, kR, P);
            const double p_new = p + div_1(v_R - v_L, k1 - k3);
            p = (p_new < 0.0) ? 0.5 * p : p_new;
        }
        if (__builtin_expect(!(p > 0x1p-300 && p < 0x1p300), 0)) return false;
        v_L = curve_q<-1>(p, u_L, p_L, c_L, GL, &kL, P);
        v_R = curve_q<+1>(p, u_R, p_R, c_R, GR, &kR, P);
        const double gap = fabs(v_L - v_R);
        if (st == 1 || st == 4) ++done;
        if (st == 3 || st == 5) ++n;
        const bool extra = CONV && st != 4 && st != 5 &&
                           (st == 0 || st == 2 ||
                            gap > fmin(CONV_ULP * (fabs(v_L) + fabs(v_R) + c_L + c_R), CONV_REL * p * fabs(k1 - k3)));
        if (st <= 1 || st == 4) {
            if (gap <= tol) {
                if (!extra) break;
                st = 4;
            } else {
                st = (gap > tol && done < GUESS_ITERS) ? 1 : 2;
            }
        } else if (gap > tol && n != N) {
            st = 3;
        } else if (extra && n != N) {
            st = 5;
        } else {
            break;
        }
    }
    // a tolerance below the velocities themselves lets the iteration end on a tiny gap
    const double share = k1 * (v_R - v_L);
    u = (__builtin_expect(tiny(v_R - v_L), 0) ? share / (k1 - k3) : div_1(share, k1 - k3)) + v_L;
    return true;
}

// Which of the waves are shocks, from the end of the Newton iteration: the
// reference asks whether v_L(q) - v_R(q) =: g(q) exceeds eps at q = p_R (the
// 3-wave) and p_L (the 1-wave), two more wave curves.  Here g(p) is known at the
// last p.  Along either curve |v'| falls with the pressure, p |v'| rises (for
// the rarefaction it is a power -nu > -1, for the shock its logarithmic slope
// lies between -1 and -1/2), and |v'| = c/(gamma p) at the side's own pressure;
// so between q and p the slope of g lies between A/pm and A/pn, where A sums
// c/gamma over the sides, pm is the largest of the three pressures and pn the
// smaller side's.  The margin M covers the rounding of the curves here and there
// (pressure ratios up to 1024).  False where that does not decide: the curves do.
// With the states behind the waves taken from the last curves (Keep) a step
// goes, at 1024^2, from .374 to .355 ms, 4096^2 learned 4.54 -> 4.34, two fluids
// 2048 x 512 .566 -> .522.
struct WaveTest {
    double A, M, g, p, pm, pn;
};
HGRP_HD bool wave_type(const WaveTest &w, double q, double eps, int &fan)
{
    const double d = w.p - q, t = d * w.A;
    const bool shock = d > 0.0 && t + (w.g - eps - w.M) * w.pm > 0.0;
    fan = !shock;
    return shock || t + (w.g - eps + w.M) * (d > 0.0 ? w.pn : w.pm) < 0.0;
}

// riemann_exact with at most N steps; kL, kR: of the curves at the star pressure
// (m = 0 where there is none).  False where the pressure leaves the range (or is
// not a number).
template <bool CONV, int N = 500>
HGRP_HD bool riemann_q(const Gas &GL, const Gas &GR, double u_L, double u_R, const Rcp &p_L, const Rcp &p_R,
                       double c_L, double c_R, double eps, double tol, double p_guess, StarQ &out, Keep &kL, Keep &kR,
                       const double *P)
{
    const bool equal = fabs(u_L - u_R) < tol && fabs(p_L.b - p_R.b) < tol;
    bool sure = false;
    kL = kR = {{0.0, 0.0}, 0.0};
    if (equal) {
        out.p = 0.5 * (p_L.b + p_R.b);
        out.u = 0.5 * (u_L + u_R);
    } else {
        double v_L = 0.0, v_R = 0.0, p;
        if (!newton_q<CONV, N>(GL, GR, u_L, u_R, p_L, p_R, c_L, c_R, tol, p_guess, p, v_L, v_R, out.u, kL, kR, P))
            return false;
        out.p = p;
        const double top = fmax(p_L.b, p_R.b);
        WaveTest w;
        w.pn = fmin(p_L.b, p_R.b);
        w.pm = fmax(top, p);
        w.p = p;
        w.g = v_L - v_R;
        w.A = c_L * GL.inv_g + c_R * GR.inv_g;
        w.M = 0x1p-46 * (fabs(u_L) + fabs(u_R) + fabs(v_L) + fabs(v_R) + eps + c_L * (GL.y_gm1 + 64.0) +
                         c_R * (GR.y_gm1 + 64.0));
        const bool s0 = wave_type(w, p_L.b, eps, out.crw0), s1 = wave_type(w, p_R.b, eps, out.crw1);
        sure = s0 && s1 && top <= 1024.0 * w.pn;
    }
    if (__builtin_expect(!sure, 0)) {
        Keep t;
        const double u_LR = curve_q<-1>(p_R.b, u_L, p_L, c_L, GL, &t, P);
        const double u_RL = curve_q<+1>(p_L.b, u_R, p_R, c_R, GR, &t, P);
        out.crw1 = (u_LR > u_R + eps) ? 0 : 1;
        out.crw0 = (u_RL > u_L - eps) ? 1 : 0;
    }
    return true;
}

// ---- the GRP solve --------------------------------------------------------------------
// The state behind a wave (rho and c next to the contact) and the speed of its
// head.  SIGN -1: the 1-wave, +1: the 3-wave.
template <int SIGN>
HGRP_HD void behind_q(double rho, double u, const Rcp &p, double c, double p_star, int fan, const Keep &k,
                      const Gas &G, double &rs, double &cs, double &speed, const double *P)
{
    if (fan) {
        Keep a = k;
        if (a.m == 0.0) {
            a.l = log_in_range(div_q(p_star, p), P);
            a.m = pow_in_range(a.l, G.mu, P);
        }
        rs = rho * pow_in_range(a.l, G.inv_g, P);
        cs = c * a.m;                                     // e_cs is mu
        speed = SIGN < 0 ? u - c : u + c;
    } else {
        rs = div_1(rho * (p_star + G.z * p.b), p.b + G.z * p_star);
        cs = sqrt_q(div_1(G.g * p_star, rs));
        const double s = c * sqrt_q(div_q(0.5 * (G.gp1() * div_q(p_star, p) + G.gm1()), {G.g, G.inv_g}));
        speed = SIGN < 0 ? u - s : u + s;
    }
}

// (1 + z) x^e_a + z x^e_b over 1 + 2 z, times TdS, minus / plus c x^e_a dI: the
// derivative along a rarefaction's characteristic; *xb receives x^e_b
template <int SIGN>
HGRP_HD double fan_line_q(double x, double c, const Gas &G, double TdS, double dI, double *xb, const double *P)
{
    const DD l = log_in_range(x, P);
    const double a = pow_in_range(l, G.e_a, P), b = pow_in_range(l, G.e_b, P);
    *xb = b;
    double d = G.opz() * a + G.z * b;
    d = div_q(d, {G.op2z(), G.y_op2z}) * TdS;
    return SIGN < 0 ? d - c * a * dI : d + c * a * dI;
}

// TdS and the Riemann invariant's derivative of a side (d_Psi for SIGN -1, d_Phi for +1)
template <int SIGN>
HGRP_HD void invariants_q(const Rcp &rho, double c, double d_rho, double d_u, double d_p, const Gas &G, double &TdS,
                          double &dI)
{
    const Rcp gm1 = {G.gm1(), G.y_gm1};
    TdS = div_q(div_q(d_p - d_rho * c * c, gm1), rho);
    const double t = div_q(div_q(div_1(G.g * d_p, c) - c * d_rho, gm1), rho);
    dI = SIGN < 0 ? d_u + t : d_u - t;
}

// One side's line of the 2x2 system for (Du/Dt, Dp/Dt) in the non-sonic case:
// a, b, d; and what the t-axis side needs again: x^e_b behind a rarefaction,
// the shock's relative speeds behind (Ss) and ahead (S).
struct LineQ {
    double a, b, d, xb, Ss, S;
};
template <int SIGN>
HGRP_HD void line_q(const Rcp &rho, double p, double c, double d_rho, double d_u, double d_p, double p_star,
                    double rs, double cs, int fan, const Gas &G, LineQ &o, const double *P)
{
    const Rcp rrs = rcp_of(rs);
    if (fan) {
        double TdS, dI;
        invariants_q<SIGN>(rho, c, d_rho, d_u, d_p, G, TdS, dI);
        o.a = 1.0;
        const double inv = recip_q(rrs);
        o.b = div_1(SIGN < 0 ? inv : -inv, cs);
        o.d = fan_line_q<SIGN>(div_1(cs, c), c, G, TdS, dI, &o.xb, P);
        o.Ss = o.S = 0.0;
    } else {
        const double ss = sqrt_q(div_q(0.5 * (G.gp1() * p + G.gm1() * p_star), rrs));
        const double s = sqrt_q(div_q(0.5 * (G.gp1() * p_star + G.gm1() * p), rho));
        const double Ss = SIGN < 0 ? -ss : ss, S = SIGN < 0 ? -s : s;
        const double q = p_star + G.z * p;
        const Rcp rq = rcp_of(q);
        const double V = sqrt_q(div_1(G.omz(), rho.b * q));
        const double H1 = div_q(0.5 * V * (p_star + G.op2z() * p), rq);
        const double H2 = div_q(-0.5 * V * (G.tpz() * p_star + G.z * p), rq);
        const double H3 = div_q(-0.5 * V * (p_star - p), rho);
        const double inv = -recip_q(rho);
        const double h = rho.b * (c * c * H2 + H3);
        const double L_p = SIGN < 0 ? inv - S * H2 : inv + S * H2;
        const double L_u = SIGN < 0 ? S + h : S - h;
        const double L_rho = SIGN < 0 ? -S * H3 : S * H3;
        const double e = rs * Ss * H1;
        o.a = SIGN < 0 ? 1.0 - e : 1.0 + e;
        const double f = div_1(Ss, rs * cs * cs);
        o.b = SIGN < 0 ? -f + H1 : -(f + H1);
        o.d = L_rho * d_rho + L_u * d_u + L_p * d_p;
        o.Ss = Ss;
        o.S = S;
        o.xb = 0.0;
    }
}

// linear_GRP_solver_Edir_Q1D at atc = eps, lambda = 0 (grp_q1d).  near2: the
// acoustic switch on the squared distance (near_threshold).  TR: with
// tangential derivatives TL, TR.  TF: two fluids, as in grp_q1d.
template <bool TRANS, bool TF, bool CONV>
HGRP_HD bool grp_q1d_q(double D[4], double U[4], const Side &L, const Side &R, const double TL[4], const double TR[4],
                       const Gas &GL, const Gas &GR, double near2, double eps, double tol, double p_guess,
                       const double *FA, double *FO, const double *P)
{
    const Rcp rL = rcp_of(L.rho), rR = rcp_of(R.rho);
    const double c_L = sqrt_q(div_q(GL.g * L.p, rL)), c_R = sqrt_q(div_q(GR.g * R.p, rR));
    const double dist2 = (L.rho - R.rho) * (L.rho - R.rho) + (L.u - R.u) * (L.u - R.u) + (L.p - R.p) * (L.p - R.p);
    const bool near = dist2 < near2;

    StarQ st;
    bool rough = false;
    double rs_L, rs_R, cs_L, cs_R, speed_L, speed_R;
    if (near) {
        st.u = 0.5 * (R.u + L.u);
        st.p = 0.5 * (R.p + L.p);
        st.crw0 = st.crw1 = 0;
        rs_L = L.rho; cs_L = c_L; speed_L = st.u - c_L;
        rs_R = R.rho; cs_R = c_R; speed_R = st.u + c_R;
    } else {
        rough = any_lane(tiny(L.u) || tiny(R.u) || tiny(L.d_u) || tiny(R.d_u));
        const Rcp pL = rcp_of(L.p), pR = rcp_of(R.p);
        Keep kL, kR;
        if (!riemann_q<CONV>(GL, GR, L.u, R.u, pL, pR, c_L, c_R, eps, tol, p_guess, st, kL, kR, P)) return false;
        behind_q<-1>(L.rho, L.u, pL, c_L, st.p, st.crw0, kL, GL, rs_L, cs_L, speed_L, P);
        behind_q<+1>(R.rho, R.u, pR, c_R, st.p, st.crw1, kR, GR, rs_R, cs_R, speed_R, P);
    }
    const double u_star = st.u, p_star = st.p;

    // the t-axis outside the fan: the upwind side's own derivative
    if (speed_L > 0.0 || speed_R < 0.0) {
        const bool left = speed_L > 0.0;
        const double rho = left ? L.rho : R.rho, u = left ? L.u : R.u, v = left ? L.v : R.v;
        const double d_rho = left ? L.d_rho : R.d_rho, d_u = left ? L.d_u : R.d_u, d_v = left ? L.d_v : R.d_v;
        const double d_p = left ? L.d_p : R.d_p, c = left ? c_L : c_R;
        const Rcp r = {rho, left ? rL.y : rR.y};
        U[0] = rho; U[1] = u; U[2] = v; U[3] = left ? L.p : R.p;
        if constexpr (TRANS) {
            const double *T = left ? TL : TR;
            D[0] = -u * d_rho - v * T[0] - rho * (d_u + T[2]);
            D[1] = -u * d_u - v * T[1] - div_q(d_p, r);
            D[2] = -u * d_v - v * T[2] - div_q(T[3], r);
            D[3] = -u * d_p - v * T[3] - rho * c * c * (d_u + T[2]);
        } else {
            D[0] = -u * d_rho - rho * d_u;
            D[1] = -u * d_u - div_q(d_p, r);
            D[2] = -u * d_v;
            D[3] = -u * d_p - rho * c * c * d_u;
        }
        if constexpr (TF) { FO[0] = left ? FA[0] : FA[2]; FO[1] = -u * (left ? FA[1] : FA[3]); }
        return true;
    }

    double C;
    if (near) {                                            // acoustic
        const bool left = u_star > 0.0;
        U[0] = left ? rs_L : rs_R; U[1] = u_star; U[2] = left ? L.v : R.v; U[3] = p_star;
        C = left ? cs_L : cs_R;
        const double z0 = U[0] * C, cc = C * C;
        const Rcp rz = rcp_of(z0), rcc = rcp_of(cc);
        const double D_p = 0.5 * ((L.d_u * z0 + L.d_p) - (R.d_u * z0 - R.d_p));
        const double D_u = 0.5 * (L.d_u + div_q(L.d_p, rz) + R.d_u - div_q(R.d_p, rz));
        const double D_v = left ? L.d_v : R.d_v;
        const double d_rho = left ? L.d_rho : R.d_rho, d_p = left ? L.d_p : R.d_p;
        const double D_rho = d_rho - div_q(d_p, rcc) + D_p / cc;
        if constexpr (TRANS) {
            const double *T = left ? TL : TR;
            const double T_p = 0.5 * ((TL[1] * z0 + TL[3]) - (TR[1] * z0 - TR[3]));
            const double T_u = 0.5 * (TL[1] + div_q(TL[3], rz) + TR[1] - div_q(TR[3], rz));
            const double T_v = T[2], T_rho = T[0] - div_q(T[3], rcc) + T_p / cc;
            D[0] = -u_star * D_rho - U[2] * T_rho - U[0] * (D_u + T_v);
            D[1] = -u_star * D_u - U[2] * T_u - D_p / U[0];
            D[2] = -u_star * D_v - U[2] * T_v - T_p / U[0];
            D[3] = -u_star * D_p - U[2] * T_p - U[0] * C * C * (D_u + T_v);
        } else {
            D[0] = -u_star * D_rho - U[0] * D_u;
            D[1] = -u_star * D_u - D_p / U[0];
            D[2] = -u_star * D_v;
            D[3] = -u_star * D_p - U[0] * C * C * D_u;
        }
        if constexpr (TF) { FO[0] = left ? FA[0] : FA[2]; FO[1] = -u_star * (left ? FA[1] : FA[3]); }
        return true;
    }

    const bool in0 = st.crw0 && u_star - cs_L > 0.0;       // the t-axis inside the 1-rarefaction
    const bool in1 = st.crw1 && u_star + cs_R < 0.0;       // inside the 3-rarefaction
    if (in0 || in1) {
        const Gas &G = in0 ? GL : GR;
        const double c = in0 ? c_L : c_R, p = in0 ? L.p : R.p, d_v = in0 ? L.d_v : R.d_v;
        const Rcp rho = {in0 ? L.rho : R.rho, in0 ? rL.y : rR.y};
        const double tc = div_q(2.0 * c, {G.gm1(), G.y_gm1});
        U[1] = G.z * (in0 ? L.u + tc : R.u - tc);
        C = in0 ? U[1] : -U[1];
        if (!(C >= 0x1p-200)) return false;                // no sonic point (a vacuum that the iteration left)
        const Rcp rC = rcp_of(C);
        const double x = div_1(C, c);
        U[3] = pow_in_range(log_in_range(x, P), G.e_sonic, P) * p;
        U[0] = div_q(div_q(G.g * U[3], rC), rC);
        U[2] = in0 ? L.v : R.v;
        double TdS, dI, xb;
        if (in0) {
            invariants_q<-1>(rho, c, L.d_rho, L.d_u, L.d_p, G, TdS, dI);
            D[1] = fan_line_q<-1>(x, c, G, TdS, dI, &xb, P);
        } else {
            invariants_q<+1>(rho, c, R.d_rho, R.d_u, R.d_p, G, TdS, dI);
            D[1] = fan_line_q<+1>(x, c, G, TdS, dI, &xb, P);
        }
        D[3] = U[0] * U[1] * D[1];
        D[0] = U[0] * U[1] * xb * TdS * G.gm1();
        D[0] = div_q(div_q(D[0] + D[3], rC), rC);
        D[2] = -U[1] * d_v * U[0] / rho.b;
        if constexpr (TF) { FO[0] = in0 ? FA[0] : FA[2]; FO[1] = -U[1] * (in0 ? FA[1] : FA[3]) * U[0] / rho.b; }
    } else {                                              // non-sonic
        LineQ l, r;
        line_q<-1>(rL, L.p, c_L, L.d_rho, L.d_u, L.d_p, p_star, rs_L, cs_L, st.crw0, GL, l, P);
        line_q<+1>(rR, R.p, c_R, R.d_rho, R.d_u, R.d_p, p_star, rs_R, cs_R, st.crw1, GR, r, P);
        const Rcp det = rcp_of(l.a * r.b - l.b * r.a);
        const double u_t = div_r(r.b * l.d - l.b * r.d, det, rough);
        const double p_t = div_r(l.a * r.d - r.a * l.d, det, rough);
        // the side of the contact that the t-axis lies on
        const bool right = u_star < 0.0;
        const double rs = right ? rs_R : rs_L;
        C = right ? cs_R : cs_L;
        const Rcp rC = rcp_of(C), rrs = rcp_of(rs), rho = {right ? R.rho : L.rho, right ? rR.y : rL.y};
        U[0] = rs; U[1] = u_star; U[2] = right ? R.v : L.v; U[3] = p_star;
        D[1] = u_t + div_r(div_r(div_r(u_star, rrs, rough), rC, rough), rC, rough) * p_t;
        D[3] = p_t + u_star * rs * u_t;
        const double c = right ? c_R : c_L, p = right ? R.p : L.p, z = right ? GR.z : GL.z;
        const double d_rho = right ? R.d_rho : L.d_rho, d_u = right ? R.d_u : L.d_u, d_p = right ? R.d_p : L.d_p;
        const double d_v = right ? R.d_v : L.d_v;
        if (right ? st.crw1 : st.crw0) {
            const double xb = right ? r.xb : l.xb;
            D[0] = div_r(rs * u_star * xb * (d_p - d_rho * c * c), rho, rough);
            D[0] = div_r(div_r(D[0] + D[3], rC, rough), rC, rough);
            D[2] = -u_star * d_v * rs / rho.b;
            if constexpr (TF) { FO[0] = right ? FA[2] : FA[0]; FO[1] = -u_star * (right ? FA[3] : FA[1]) * rs / rho.b; }
        } else {
            const double Ss = right ? r.Ss : l.Ss, S = right ? r.S : l.S;
            const Rcp rV = rcp_of(p + z * p_star), rSs = rcp_of(Ss);
            const double H1 = div_q(div_q(rho.b * p * (1.0 - z * z), rV), rV);
            const double H2 = div_q(div_q(rho.b * p_star * (z * z - 1.0), rV), rV);
            const double H3 = div_q(p_star + z * p, rV);
            const double L_rho = S * H3 * d_rho;
            const double L_u = -rho.b * (H2 * c * c + H3) * d_u;
            const double L_p = H2 * S * d_p;
            D[0] = (div_q(div_q(u_star + Ss, rC), rC) - u_star * H1) * p_t + rs * u_star * Ss * H1 * u_t;
            D[0] = div_r(D[0] - u_star * (L_p + L_rho + L_u), rSs, rough);
            // the reference adds lambda times a derivative over S + u here: nothing but NaN where that is zero
            if (S + (right ? R.u : L.u) == 0.0) D[0] = NAN;
            D[2] = -u_star * S * d_v / Ss;
            if constexpr (TF) { FO[0] = right ? FA[2] : FA[0]; FO[1] = -u_star * S * (right ? FA[3] : FA[1]) / Ss; }
        }
    }
    if constexpr (TRANS) {
        const bool left = u_star > 0.0;
        const double *T = left ? TL : TR;
        const double z0 = U[0] * C, cc = C * C;
        const Rcp rz = rcp_of(z0), rcc = rcp_of(cc);
        const double T_p = 0.5 * ((TL[1] * z0 + TL[3]) - (TR[1] * z0 - TR[3]));
        const double T_u = 0.5 * (TL[1] + div_q(TL[3], rz) + TR[1] - div_q(TR[3], rz));
        const double T_rho = T[0] - div_q(T[3], rcc) + T_p / cc;
        D[0] = D[0] - U[2] * T_rho - U[0] * T[2];
        D[1] = D[1] - U[2] * T_u;
        D[2] = D[2] - U[2] * T[2] - T_p / U[0];
        D[3] = D[3] - U[2] * T_p - U[0] * C * C * T[2];
    }
    return true;
}

// ---- the flux -------------------------------------------------------------------------
// The acoustic switch sqrt(d) < eps on d itself: the smallest double whose
// root is not below eps (the rounded root grows with its argument).
inline double near_threshold(double eps)
{
    if (!(eps > 0.0)) return 0.0;               // nothing is below it
    if (!(eps < INFINITY)) return eps;
    double t = eps * eps;
    if (!(t < INFINITY)) return INFINITY;
    while (t > 0.0 && sqrt(t) >= eps) t = nextafter(t, 0.0);
    while (sqrt(t) < eps) t = nextafter(t, INFINITY);
    return t;
}

// GRP_2D_flux in the split sweeps (grp_2d_flux<DIR, CONV>; *code its return
// value).  False, with nothing written, where the interface is not in range.
template <int DIR, bool CONV>
__device__ __forceinline__ bool flux_split_q(const Side &L, const Side &R, const Gas &G, double near2, double tau,
                                             double eps, double F[4], double I[4], double tol, double p_guess,
                                             int *code, const double *P)
{
    if (!(gas_in_range(G) && sides_in_range(L, R))) return false;
    Side l = L, r = R;
    if constexpr (DIR == 1) {                    // into the interface's frame
        l.u = L.v; l.v = -L.u; l.d_u = L.d_v; l.d_v = -L.d_u;
        r.u = R.v; r.v = -R.u; r.d_u = R.d_v; r.d_v = -R.d_u;
    }
    double D[4], U[4];
    if (!grp_q1d_q<false, false, CONV>(D, U, l, r, nullptr, nullptr, G, G, near2, eps, tol, p_guess, nullptr, nullptr, P))
        return false;
    *code = flux_from_mid<DIR>(U, D, G, tau, eps, F, I);
    return true;
}

// GRP_2D_flux in the unsplit step (grp_2d_flux_n: one gas, tangential
// derivatives in grid axes), normal x (dir 0) or y (dir 1).
template <bool CONV>
__device__ __forceinline__ bool flux_transversal_q(const Side &L, const Side &R, const double TL[4], const double TR[4],
                                                   const Gas &G, int dir, double near2, double tau, double eps, double F[4],
                                                   double I[4], double tol, double p_guess, int *code, const double *P)
{
    const double t = ((fabs(TL[0]) + fabs(TL[1])) + (fabs(TL[2]) + fabs(TL[3]))) +
                     ((fabs(TR[0]) + fabs(TR[1])) + (fabs(TR[2]) + fabs(TR[3])));
    if (!(gas_in_range(G) && sides_in_range(L, R) && t <= MOST)) return false;
    Side l = L, r = R;
    double tl[4] = {TL[0], TL[1], TL[2], TL[3]}, tr[4] = {TR[0], TR[1], TR[2], TR[3]};
    if (dir) {                                   // into the interface's frame
        l.u = L.v; l.v = -L.u; l.d_u = L.d_v; l.d_v = -L.d_u;
        r.u = R.v; r.v = -R.u; r.d_u = R.d_v; r.d_v = -R.d_u;
        tl[1] = TL[2]; tl[2] = -TL[1];
        tr[1] = TR[2]; tr[2] = -TR[1];
    }
    double D[4], U[4];
    if (!grp_q1d_q<true, false, CONV>(D, U, l, r, tl, tr, G, G, near2, eps, tol, p_guess, nullptr, nullptr, P)) return false;
    *code = flux_from_mid_n(U, D, G, dir ? 0.0 : 1.0, dir ? 1.0 : 0.0, tau, eps, F, I);
    return true;
}

// ---- two fluids --------------------------------------------------------------------
// mix_gamma, gas_of: a fraction is divided by constants, and what a tiny one's
// quotient may be off by is lost in the sum
__device__ __forceinline__ double mix_inv_gm1_q(double fa, const TwoGas &T)
{
    return div_q(fa, {T.a.gm1(), T.a.y_gm1}) + div_q(1.0 - fa, {T.b.gm1(), T.b.y_gm1});
}
__device__ __forceinline__ double mix_gamma_q(double fa, const TwoGas &T) { return recip_1(mix_inv_gm1_q(fa, T)) + 1.0; }

__device__ __forceinline__ Gas make_gas_q(double g)      // make_gas for gas_in_range(g)
{
    const double gm1 = g - 1.0, gp1 = g + 1.0;
    Rcp rg = rcp_of(g), rm = rcp_of(gm1);
    rg.y = recip_q(rg);
    rm.y = recip_q(rm);
    const Rcp r2g = {2.0 * g, 0.5 * rg.y};
    Gas s;
    s.g = g;
    s.mu = div_q(gm1, r2g);
    s.nu = div_q(gp1, r2g);
    s.z = div_1(gm1, gp1);
    s.inv_g = rg.y;
    s.e_cs = s.mu;                               // 0.5 (g-1) / g, the same quotient
    s.e_sonic = div_q(2.0 * g, rm);
    const Rcp rz = rcp_of(s.z);
    s.e_a = div_q(0.5, rz);
    s.e_b = div_q(1.0 + s.z, rz);
    s.g_gm1 = div_q(g, rm);
    s.y_gm1 = rm.y;
    s.y_op2z = recip_1(s.op2z());
    return s;
}
__device__ __forceinline__ bool two_in_range(const TwoGas &T)
{
    return T.a.gm1() >= 0x1p-20 && T.a.g <= 0x1p20 && T.b.gm1() >= 0x1p-20 && T.b.g <= 0x1p20;
}

// GRP_2D_flux with two fluids (grp_2d_flux_tf).
template <int DIR, bool CONV>
__device__ __forceinline__ bool flux_two_fluid_q(const Side &L, const Side &R, const TwoGas &T, const double FA[4],
                                                 double near2, double tau, double eps, double F[4], double I[4],
                                                 double FZ[3], double tol, double p_guess, int *code, const double *P)
{
    constexpr double n_x = DIR == 0 ? 1.0 : 0.0, n_y = DIR == 0 ? 0.0 : 1.0;
    // reconstructed fractions leave [0, 1] by rounding only
    const bool fr = FA[0] >= -0.5 && FA[0] <= 1.5 && FA[2] >= -0.5 && FA[2] <= 1.5 &&
                    fabs(FA[1]) + fabs(FA[3]) <= 0x1p100;
    if (!(fr && two_in_range(T) && sides_in_range(L, R))) return false;
    const bool pure_L = FA[0] == 1.0 || FA[0] == 0.0, pure_R = FA[2] == 1.0 || FA[2] == 0.0;
    Gas GL = FA[0] == 1.0 ? T.a : T.b, GR = FA[2] == 1.0 ? T.a : T.b;
    if (!pure_L) GL = make_gas_q(mix_gamma_q(FA[0], T));
    if (!pure_R) GR = make_gas_q(mix_gamma_q(FA[2], T));
    if (!(gas_in_range(GL) && gas_in_range(GR))) return false;
    Side l = L, r = R;
    if constexpr (DIR == 1) {
        l.u = L.v; l.v = -L.u; l.d_u = L.d_v; l.d_v = -L.d_u;
        r.u = R.v; r.v = -R.u; r.d_u = R.d_v; r.d_v = -R.d_u;
    }
    double dire[4], mid[4], fo[2];
    if (!grp_q1d_q<false, true, CONV>(dire, mid, l, r, nullptr, nullptr, GL, GR, near2, eps, tol, p_guess, FA, fo, P))
        return false;
    *code = star_dire_bad(mid, dire, eps);
    if (*code) {
        F[0] = F[1] = F[2] = F[3] = 0.0;
        I[0] = I[1] = I[2] = I[3] = 0.0;
        FZ[0] = FZ[1] = FZ[2] = 0.0;
        return true;
    }
    const double rho_mid = mid[0] + 0.5 * tau * dire[0];
    const double u_mid = (mid[1] + 0.5 * tau * dire[1]) * n_x - (mid[2] + 0.5 * tau * dire[2]) * n_y;
    const double v_mid = (mid[1] + 0.5 * tau * dire[1]) * n_y + (mid[2] + 0.5 * tau * dire[2]) * n_x;
    const double p_mid = mid[3] + 0.5 * tau * dire[3];
    const double a_mid = fo[0] + 0.5 * tau * fo[1];
    double ge = a_mid == 1.0 ? T.a.g_gm1 : T.b.g_gm1;
    if (!(a_mid == 1.0 || a_mid == 0.0)) {
        if (a_mid >= -0.5 && a_mid <= 1.5) {
            const double gamma_mid = mix_gamma_q(a_mid, T);
            ge = div_1(gamma_mid, gamma_mid - 1.0);
        } else {
            const double gamma_mid = mix_gamma(a_mid, T);
            ge = gamma_mid / (gamma_mid - 1.0);
        }
    }
    F[0] = rho_mid * (u_mid * n_x + v_mid * n_y);
    F[1] = F[0] * u_mid + p_mid * n_x;
    F[2] = F[0] * v_mid + p_mid * n_y;
    F[3] = ge * p_mid / rho_mid + 0.5 * (u_mid * u_mid + v_mid * v_mid);
    F[3] = F[0] * F[3];
    I[1] = (mid[1] + tau * dire[1]) * n_x - (mid[2] + tau * dire[2]) * n_y;
    I[2] = (mid[1] + tau * dire[1]) * n_y + (mid[2] + tau * dire[2]) * n_x;
    I[0] = mid[0] + tau * dire[0];
    I[3] = mid[3] + tau * dire[3];
    const double un_mid = u_mid * n_x + v_mid * n_y;
    FZ[0] = un_mid * a_mid;
    FZ[1] = un_mid;
    FZ[2] = fo[0] + tau * fo[1];
    return true;
}

}  // namespace hgrp
