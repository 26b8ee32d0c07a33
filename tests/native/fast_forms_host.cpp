// Host build of the forms of the steps' interface solver (hydrocode-fusion_amd/csrc/grp_fast.hpp,
// g2d_device.hpp) that the unsplit step and the two-fluid sweeps run, each in both stopping rules and
// from a given starting pressure, beside the IEEE solver on the same interfaces.
#include <hip/hip_runtime.h>
#include "g2d_device.hpp"

using namespace hgrp;

static Side side_of(const double *l) { return {l[3], l[4], l[5], l[6], l[7], l[8], l[9], l[10]}; }

// The unsplit step's flux.  L, R: sides of 15 doubles; guess: starting pressures (<= 0: none).
// Rows of code F I; returns how many interfaces the fast solver took (the others' fast rows: NaN code).
template <bool CONV>
static int transversal(const double *L, const double *R, int n, double tau, double eps, double tol, int dir,
                       const double *guess, double *fast, double *ieee)
{
    int took = 0;
    for (int k = 0; k < n; ++k) {
        const double *l = L + 15 * k, *r = R + 15 * k;
        const Side a = side_of(l), b = side_of(r);
        const Gas G = make_gas(l[0]);
        double *f = fast + 9 * k, *o = ieee + 9 * k;
        o[0] = grp_2d_flux_n<CONV>(a, b, l + 11, r + 11, G, dir ? 0.0 : 1.0, dir ? 1.0 : 0.0, tau, eps, o + 1, o + 5,
                                   tol, guess[k]);
        int code = 0;
        const bool ok = flux_transversal_q<CONV>(a, b, l + 11, r + 11, G, dir, near_threshold(eps), tau, eps, f + 1,
                                                 f + 5, tol, guess[k], &code, powtab::TAB);
        f[0] = ok ? code : NAN;
        took += ok;
    }
    return took;
}
extern "C" int ff_transversal(const double *L, const double *R, int n, double tau, double eps, double tol, int dir,
                              int conv, const double *guess, double *fast, double *ieee)
{
    return conv ? transversal<true>(L, R, n, tau, eps, tol, dir, guess, fast, ieee)
                : transversal<false>(L, R, n, tau, eps, tol, dir, guess, fast, ieee);
}

// The two-fluid flux: FA = {a_L, d_a_L, a_R, d_a_R} per interface.  Rows of code F I Z (12).
template <int DIR, bool CONV>
static int two_fluid(const double *L, const double *R, const double *FA, int n, double tau, double eps, double tol,
                     double ga, double gb, const double *guess, double *fast, double *ieee)
{
    int took = 0;
    TwoGas T;
    T.a = make_gas(ga);
    T.b = make_gas(gb);
    for (int k = 0; k < n; ++k) {
        const Side a = side_of(L + 15 * k), b = side_of(R + 15 * k);
        const double *fa = FA + 4 * k;
        double *f = fast + 12 * k, *o = ieee + 12 * k;
        o[0] = grp_2d_flux_tf<DIR, CONV>(a, b, T, fa, tau, eps, o + 1, o + 5, o + 9, tol, guess[k]);
        int code = 0;
        const bool ok = flux_two_fluid_q<DIR, CONV>(a, b, T, fa, near_threshold(eps), tau, eps, f + 1, f + 5, f + 9, tol,
                                                    guess[k], &code, powtab::TAB);
        f[0] = ok ? code : NAN;
        took += ok;
    }
    return took;
}
extern "C" int ff_two_fluid(const double *L, const double *R, const double *FA, int n, double tau, double eps, double tol,
                            int dir, int conv, double ga, double gb, const double *guess, double *fast, double *ieee)
{
    if (dir == 0)
        return conv ? two_fluid<0, true>(L, R, FA, n, tau, eps, tol, ga, gb, guess, fast, ieee)
                    : two_fluid<0, false>(L, R, FA, n, tau, eps, tol, ga, gb, guess, fast, ieee);
    return conv ? two_fluid<1, true>(L, R, FA, n, tau, eps, tol, ga, gb, guess, fast, ieee)
                : two_fluid<1, false>(L, R, FA, n, tau, eps, tol, ga, gb, guess, fast, ieee);
}

// G2D with its star state from the fast solve (and from the IEEE one where that is out of its range) beside
// the IEEE form.  Sides of 21 doubles; rows of ws D U U_star (20).  Returns how many interfaces come with
// both sides in the fast solve's range.
template <bool CONV>
static int g2d(const double *L, const double *R, int n, double eps, double tol, const double *guess, double *fast,
               double *ieee)
{
    int in = 0;
    for (int k = 0; k < n; ++k) {
        const double *l = L + 21 * k, *r = R + 21 * k;
        const G2Side a = g2_side_of(l, -1.0), b = g2_side_of(r, 1.0);
        in += fmin(a.p, b.p) >= LEAST && a.p + b.p <= MOST && fmin(a.c, b.c) >= LEAST &&
              fabs(a.u) + fabs(b.u) + a.c + b.c <= MOST && gas_in_range(a.G) && gas_in_range(b.G);
        double *f = fast + 20 * k, *o = ieee + 20 * k;
        grp_g2d<CONV, true>(f + 2, f + 8, f, f + 14, a, b, l[1], r[2], eps, eps, tol, guess[k], powtab::TAB);
        grp_g2d<CONV, false>(o + 2, o + 8, o, o + 14, a, b, l[1], r[2], eps, eps, tol, guess[k]);
    }
    return in;
}
extern "C" int ff_g2d(const double *L, const double *R, int n, double eps, double tol, int conv, const double *guess,
                      double *fast, double *ieee)
{
    return conv ? g2d<true>(L, R, n, eps, tol, guess, fast, ieee) : g2d<false>(L, R, n, eps, tol, guess, fast, ieee);
}
