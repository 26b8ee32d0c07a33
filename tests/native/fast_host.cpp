// Host build of the steps' interface solver (hydrocode-fusion_amd/csrc/grp_fast.hpp) beside the
// IEEE solver it stands in for (grp_device.hpp), on the same interfaces.
#include <hip/hip_runtime.h>
#include "grp_fast.hpp"

using namespace hgrp;

// L, R: sides of 15 doubles; conv: the converge rule at tol 1e-12; guess: starting pressures (<= 0: none).
// fast, ieee: rows of code F I; returns how many interfaces the fast solver took
// (the others' fast rows are left alone).
template <int DIR, bool CONV>
static int both(const double *l, const double *r, double tau, double eps, double tol, double guess, double *fast,
                double *ieee)
{
    const Side a{l[3], l[4], l[5], l[6], l[7], l[8], l[9], l[10]}, b{r[3], r[4], r[5], r[6], r[7], r[8], r[9], r[10]};
    const Gas G = make_gas(l[0]);
    double F[4] = {0, 0, 0, 0}, I[4] = {0, 0, 0, 0};
    ieee[0] = grp_2d_flux<DIR, CONV>(a, b, G, tau, eps, F, I, tol, guess);
    for (int q = 0; q < 4; ++q) { ieee[1 + q] = F[q]; ieee[5 + q] = I[q]; }
    int code = 0;
    if (!flux_split_q<DIR, CONV>(a, b, G, near_threshold(eps), tau, eps, F, I, tol, guess, &code)) return 0;
    fast[0] = code;
    for (int q = 0; q < 4; ++q) { fast[1 + q] = F[q]; fast[5 + q] = I[q]; }
    return 1;
}

extern "C" int fh_split_many(const double *L, const double *R, int n, double tau, double eps, int dir, int conv,
                             const double *guess, double *fast, double *ieee)
{
    int took = 0;
    for (int k = 0; k < n; ++k) {
        const double *l = L + 15 * k, *r = R + 15 * k;
        double *f = fast + 9 * k, *i = ieee + 9 * k;
        const double tol = conv ? 1e-12 : eps;
        if (dir == 0)
            took += conv ? both<0, true>(l, r, tau, eps, tol, guess[k], f, i) : both<0, false>(l, r, tau, eps, tol, guess[k], f, i);
        else
            took += conv ? both<1, true>(l, r, tau, eps, tol, guess[k], f, i) : both<1, false>(l, r, tau, eps, tol, guess[k], f, i);
    }
    return took;
}

extern "C" double fh_near_threshold(double eps) { return near_threshold(eps); }
