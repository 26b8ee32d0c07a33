// grp1d_fast.hpp -- the 1D ensemble's interface solver in the arithmetic of
// fast_arith.hpp: grp_edir (grp1d_device.hpp) at atc = eps, bit for bit (a
// zero's sign aside), for sides far from the ends of the exponent range (slopes
// of density and pressure zero or differences of such values over h).  The
// star state, the reciprocals and the treatment of tiny velocities are those of
// grp_fast.hpp; a shock's speed is formed once.
#pragma once
#include "grp1d_device.hpp"
#include "grp_fast.hpp"

namespace hgrp {

HGRP_HD bool sides1_in_range(const Side1 &L, const Side1 &R)
{
    const double m = ((fabs(L.u) + fabs(R.u)) + (fabs(L.s_rho) + fabs(R.s_rho))) +
                     ((fabs(L.s_u) + fabs(R.s_u)) + (fabs(L.s_p) + fabs(R.s_p)));      // NaN for a NaN
    return L.rho >= LEAST && L.p >= LEAST && R.rho >= LEAST && R.p >= LEAST &&
           fmax(fmax(L.rho, L.p), fmax(R.rho, R.p)) <= MOST && m <= MOST;
}

// the axis inside the rarefaction next to side S (grp_edir's sonic branches)
// false where there is no sonic point (a vacuum that the iteration left)
template <int SIGN>
HGRP_HD bool edir_sonic_q(double D[3], double U[3], const Side1 &S, const Rcp &rho, double c, const Gas &G, const double *P)
{
    const Rcp gm1 = {G.gm1(), G.y_gm1}, rg = {G.g, G.inv_g};
    const double t = div_q(2.0 * c, gm1);
    U[1] = G.z * (SIGN < 0 ? S.u + t : S.u - t);
    if (!((SIGN < 0 ? U[1] : -U[1]) >= 0x1p-200)) return false;
    U[2] = div_1(div_q(U[1] * U[1] * S.rho, rg), pow_in_range(log_in_range(S.p, P), G.inv_g, P));
    U[2] = pow_in_range(log_in_range(U[2], P), G.g_gm1, P);
    const Rcp rU = rcp_of(U[1]);
    U[0] = div_q(div_q(G.g * U[2], rU), rU);
    const DD l = log_in_range(div_1(SIGN < 0 ? U[1] : -U[1], c), P);
    const double pw_a = pow_in_range(l, G.e_a, P), pw_b = pow_in_range(l, G.e_b, P);
    const double e = S.s_p - S.s_rho * c * c;
    D[1] = div_q(0.5 * (pw_a * (1.0 + G.z) + pw_b * G.z), {0.5 + G.z, 2.0 * G.y_op2z});
    D[1] = div_q(div_q(D[1] * e, gm1), rho);
    const double r = div_q(div_q(div_1(G.g * S.s_p, c) - c * S.s_rho, gm1), rho);
    D[1] = SIGN < 0 ? D[1] - c * pw_a * (S.s_u + r) : D[1] + c * pw_a * (S.s_u - r);
    D[2] = U[0] * U[1] * D[1];
    D[0] = div_q(U[0] * U[1] * pw_b * e, rho);
    D[0] = div_q(div_q(D[0] + D[2], rU), rU);
    return true;
}

// one side's row a u_t + b p_t = d in the non-sonic case; pw_b as in grp_edir
template <int SIGN>
HGRP_HD void edir_row_q(const Side1 &S, const Rcp &rho, double c, double p_star, double u_star, const Rcp &rs, const Rcp &cs,
                        int fan, double shk, const Gas &G, double &a, double &b, double &d, double &pw_b, const double *P)
{
    if (fan) {
        const Rcp gm1 = {G.gm1(), G.y_gm1};
        a = 1.0;
        const double inv = recip_q(rs);
        b = div_q(SIGN < 0 ? inv : -inv, cs);
        const Rcp rc = rcp_of(c);
        const DD l = log_in_range(div_q(cs.b, rc), P);
        const double pw_a = pow_in_range(l, G.e_a, P);
        pw_b = pow_in_range(l, G.e_b, P);
        d = div_q(0.5 * (pw_a * (1.0 + G.z) + pw_b * G.z), {0.5 + G.z, 2.0 * G.y_op2z});
        d = div_q(div_q(d * (S.s_p - S.s_rho * c * c), gm1), rho);
        const double r = div_q(div_q(div_q(G.g * S.s_p, rc) - c * S.s_rho, gm1), rho);
        d = SIGN < 0 ? d - c * pw_a * (S.s_u + r) : d + c * pw_a * (S.s_u - r);
    } else {
        const double z = G.z, q = p_star + z * S.p;
        const Rcp rq = rcp_of(q);
        const double V = sqrt_q(div_1(1.0 - z, S.rho * q));
        const double H1 = div_q(0.5 * V * (p_star + G.op2z() * S.p), rq);
        const double H2 = div_q(-0.5 * V * (G.tpz() * p_star + z * S.p), rq);
        const double H3 = div_q(-0.5 * V * (p_star - S.p), rho);
        const double m = rs.b * (shk - u_star) * H1, e = div_q(div_q(div_q(u_star - shk, rs), cs), cs);
        a = SIGN < 0 ? 1.0 - m : 1.0 + m;
        b = SIGN < 0 ? e + H1 : e - H1;
        const double inv = recip_q(rho);
        const double w = SIGN < 0 ? S.u - shk : shk - S.u;
        const double L_u = SIGN < 0 ? shk - S.u + S.rho * c * c * H2 + S.rho * H3 : shk - S.u - S.rho * c * c * H2 - S.rho * H3;
        d = w * H3 * S.s_rho + L_u * S.s_u + (w * H2 - inv) * S.s_p;
        pw_b = 0.0;
    }
}

// near2: the acoustic switch on the squared distance; c_L, c_R: sqrt(gamma p / rho).
// False, with nothing to use, where the interface is for grp_edir.
HGRP_HD bool grp_edir_q(double D[3], double U[3], const Side1 &L, const Side1 &R, const Rcp &rL, const Rcp &rR, double c_L,
                        double c_R, const Gas &G, double near2, double eps, const double *P)
{
    const double dist2 = (L.u - R.u) * (L.u - R.u) + (L.p - R.p) * (L.p - R.p);
    if (dist2 < near2) {
        if (L.u - c_L > 0.0) { edir_upwind(D, U, L.rho, L.u, L.p, L.s_rho, L.s_u, L.s_p, G); return true; }
        if (R.u + c_R < 0.0) { edir_upwind(D, U, R.rho, R.u, R.p, R.s_rho, R.s_u, R.s_p, G); return true; }
        const double u = 0.5 * (R.u + L.u), p = 0.5 * (R.p + L.p), m = u - c_L;
        if (m == 0.0) return false;
        const Rcp qL = rcp_of(c_L), qR = rcp_of(c_R);
        const double PI = div_q(div_q(div_q(div_1((u + c_R) * L.rho * c_L * c_L, m), rR), qR), qR);
        const double kL = div_q(L.s_p, rL), kR = div_q(R.s_p, rR);
        // velocities' tails (see sides_in_range) are divided by IEEE division from here on
        D[1] = (kL + c_L * L.s_u) * PI / (1.0 - PI) + (kR - c_R * R.s_u) / (PI - 1.0);
        D[2] = div_q(div_q(div_q(u + c_R, rR), qR), qR) - div_q(div_q(div_q(m, rL), qL), qL);
        D[2] = (kR - c_R * R.s_u - kL - c_L * L.s_u) / D[2];
        const bool left = u > 0.0;
        const double rs = left ? L.rho : R.rho, cs = left ? c_L : c_R;
        const Rcp q = {cs, left ? qL.y : qR.y};
        U[0] = rs; U[1] = u; U[2] = p;
        D[2] = D[2] * (1.0 - div_q(div_q(u * u, q), q)) + rs * u * D[1];
        D[0] = (u * ((left ? L.s_p : R.s_p) - (left ? L.s_rho : R.s_rho) * cs * cs) + D[2]) / cs / cs;
        return true;
    }

    const bool rough = any_lane(tiny(L.u) || tiny(R.u) || tiny(L.s_u) || tiny(R.s_u));
    const Rcp pL = rcp_of(L.p), pR = rcp_of(R.p);
    StarQ st;
    Keep wL, wR;
    if (!riemann_q<false, 50>(G, G, L.u, R.u, pL, pR, c_L, c_R, eps, eps, -1.0, st, wL, wR, P)) return false;
    const double u = st.u, p = st.p, z = G.z;
    const double rs_L = p > L.p ? div_1(L.rho * (p + z * L.p), L.p + z * p)
                                : L.rho * pow_in_range(wL.m != 0.0 ? wL.l : log_in_range(div_q(p, pL), P), G.inv_g, P);
    const double rs_R = p > R.p ? div_1(R.rho * (p + z * R.p), R.p + z * p)
                                : R.rho * pow_in_range(wR.m != 0.0 ? wR.l : log_in_range(div_q(p, pR), P), G.inv_g, P);
    const Rcp qL = rcp_of(rs_L), qR = rcp_of(rs_R);
    const Rcp kL = rcp_of(sqrt_q(div_q(G.g * p, qL))), kR = rcp_of(sqrt_q(div_q(G.g * p, qR)));
    // shock speeds; where the density does not change by an ulp the quotient is IEEE's infinity or NaN
    if ((!st.crw0 && rs_L == L.rho) || (!st.crw1 && rs_R == R.rho)) return false;
    const double s_L = st.crw0 ? L.u - c_L : div_r(rs_L * u - L.rho * L.u, rcp_of(rs_L - L.rho), rough);
    const double s_R = st.crw1 ? R.u + c_R : div_r(rs_R * u - R.rho * R.u, rcp_of(rs_R - R.rho), rough);

    if (s_L > 0.0) {
        const double v = L.u;
        D[0] = -L.s_rho * v - L.rho * L.s_u;
        D[1] = (D[0] * v + L.s_rho * v * v + 2.0 * L.rho * v * L.s_u + L.s_p) / -L.rho;
        D[2] = -div_r((L.s_u * L.p + v * L.s_p) * G.g, {G.gm1(), G.y_gm1}, rough) - 0.5 * L.s_rho * v * v * v
               - 1.5 * L.rho * v * v * L.s_u;
        D[2] = D[2] - 0.5 * D[0] * v * v - L.rho * v * D[1];
        D[2] = D[2] * (G.g - 1.0);
        U[0] = L.rho; U[1] = L.u; U[2] = L.p;
        return true;
    }
    if (s_R < 0.0) { edir_upwind(D, U, R.rho, R.u, R.p, R.s_rho, R.s_u, R.s_p, G); return true; }
    if (st.crw0 && u - kL.b > 0.0) return edir_sonic_q<-1>(D, U, L, rL, c_L, G, P);
    if (st.crw1 && u + kR.b < 0.0) return edir_sonic_q<+1>(D, U, R, rR, c_R, G, P);

    double a_L, b_L, d_L, w_L, a_R, b_R, d_R, w_R;
    edir_row_q<-1>(L, rL, c_L, p, u, qL, kL, st.crw0, s_L, G, a_L, b_L, d_L, w_L, P);
    edir_row_q<+1>(R, rR, c_R, p, u, qR, kR, st.crw1, s_R, G, a_R, b_R, d_R, w_R, P);
    const Rcp ra = rcp_of(a_L);
    const double p_t = div_r(div_r(d_L * a_R, ra, rough) - d_R, rcp_of(div_q(b_L * a_R, ra) - b_R), rough);
    const double u_t = div_r(d_L - b_L * p_t, ra, rough);
    // the side of the contact that the axis lies on
    const bool right = u < 0.0;
    const Side1 &S = right ? R : L;
    const double rho = S.rho, ps = S.p, us = S.u, s_rho = S.s_rho, s_u = S.s_u, s_p = S.s_p, c = right ? c_R : c_L;
    const Rcp rs = {right ? rs_R : rs_L, right ? qR.y : qL.y}, cs = {right ? kR.b : kL.b, right ? kR.y : kL.y};
    const Rcp rr = {rho, right ? rR.y : rL.y};
    U[0] = rs.b; U[1] = u; U[2] = p;
    D[1] = u_t + div_r(div_r(div_r(u * p_t, rs, rough), cs, rough), cs, rough);
    D[2] = p_t + rs.b * u * u_t;
    if (right ? st.crw1 : st.crw0) {
        D[0] = div_r(rs.b * u * (right ? w_R : w_L) * (s_p - s_rho * c * c), rr, rough);
        D[0] = div_r(div_r(D[0] + D[2], cs, rough), cs, rough);
    } else {
        const double shk = right ? s_R : s_L, g_rho = u - shk;
        if (g_rho == 0.0) return false;
        const Rcp rV = rcp_of(ps + z * p);
        const double H1 = div_q(div_q(rho * ps * G.omzz(), rV), rV);
        const double H2 = div_q(div_q(rho * p * G.zzm1(), rV), rV);
        const double H3 = div_q(p + z * ps, rV);
        const double g_u = u * rs.b * (shk - u) * H1;
        const double g_p = div_r(div_r(shk, cs, rough), cs, rough) - u * H1;
        const double f = (shk - us) * (H2 * s_p + H3 * s_rho) - rho * (H2 * c * c + H3) * s_u;
        D[0] = div_r(f * u - g_p * p_t - g_u * u_t, rcp_of(g_rho), rough);
    }
    return true;
}

}  // namespace hgrp
