// fast_arith.hpp -- IEEE division and square root in FP64 without the range
// scaling, for operands known to be in range.
//
// What hipcc emits for a / b and sqrt(x) first scales the operands
// (v_div_scale, v_ldexp with its compares) and fixes the result up at the end,
// so that denormals, overflow and infinities come out right: 11 and 18
// instructions besides the seed.  Where the caller knows that the operands are
// far from the ends of the exponent range the same refinement without them
// gives the same double: the scaling is by powers of two, and the last step
// rounds the exact remainder's correction (Markstein).  A quotient is then 3
// operations once the divisor's reciprocal is known, and several quotients by
// one divisor share it (Rcp); a fresh reciprocal is the seed and 4 operations,
// a square root the seed and 9.  A root that is a divisor takes a reciprocal of
// its own: what the root's steps leave of 1/sqrt(x) is not rounded right for a
// root just below a power of two (1/(2 - j 2^-52) lies j^2 2^-107 above the
// middle of two doubles for odd j), and some quotients by it end an ulp off.
//
// In range means: divisors and radicands in [2^-700, 2^700], numerators zero
// or in [2^-900, 2^900], quotients in [2^-900, 2^900].  The quotient of a zero
// has the sign of IEEE division for a positive divisor.
#pragma once
#include <math.h>

#include "fastpow.hpp"

namespace hgrp {

// The seeds: within 2^-24.3 of 1/b (4e9 values on gfx950), and rounded where b
// is one ulp below a power of two, the one b that the steps below could not put
// right.  A host build's are as rough, but rounded over the few b just below a
// power of two for which two steps from a rough one may end an ulp off (there
// the device's IEEE division takes the same steps, the host's does not).
HGRP_HD double rcp_seed(double b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcp(b);
#else
    int e;
    return fabs(frexp(b, &e)) > 1.0 - 0x1p-47 ? 1.0 / b : 1.0 / b * (1.0 + 0x1.3p-25);
#endif
}
HGRP_HD double rsq_seed(double x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rsq(x);
#else
    return 1.0 / sqrt(x) * (1.0 - 0x1.3p-25);
#endif
}

// A divisor b with y = 1/b, as IEEE division forms it.  Two Newton steps leave y
// within 2^-95 of 1/b before its rounding: that is the rounded reciprocal
// except where 1/b lies that close to the middle of two doubles, as it does for
// every other b just below 1 (1 in 100 there).  A quotient's last step makes up
// for it (no quotient by 16 M such b was off on gfx950, nor was the IEEE
// division's, which takes the same steps); a reciprocal that is a result takes
// that step too (recip_q).
struct Rcp {
    double b, y;
};
HGRP_HD Rcp rcp_of(double b)
{
    double y = rcp_seed(b);
    y = fma(y, fma(-b, y, 1.0), y);
    y = fma(y, fma(-b, y, 1.0), y);
    return {b, y};
}

// a / r.b
HGRP_HD double div_q(double a, const Rcp &r)
{
    const double q = a * r.y;
    return fma(-fma(q, r.b, -a), r.y, q);
}
HGRP_HD double recip_q(const Rcp &r) { return fma(-fma(r.y, r.b, -1.0), r.y, r.y); }
HGRP_HD double recip_1(double b) { return recip_q(rcp_of(b)); }
HGRP_HD double div_1(double a, double b) { return div_q(a, rcp_of(b)); }

HGRP_HD double sqrt_q(double x)
{
    const double y = rsq_seed(x);
    double s = x * y, h = 0.5 * y;
    const double r = fma(-h, s, 0.5);
    h = fma(h, r, h);
    s = fma(s, r, s);
    s = fma(fma(-s, s, x), h, s);
    return fma(fma(-s, s, x), h, s);
}

// log_dd and exp_dd (fastpow.hpp) with every operation that changes nothing
// left out: a sum whose larger term is known takes the 3-operation error term
// (exact either way), products that are exact go into an FMA, and the result
// is the same double-double.  The table index is masked, so that a base out of
// range reads inside the table.  The logarithm of 1 is (0, ~1e-19), whose
// exponential rounds to 1.
HGRP_HD DD fast_sum(double a, double b)      // |a| >= |b| or a == 0
{
    const double s = a + b;
    return {s, b - (s - a)};
}

// The pow functions below take the tables (powtab::TAB or a copy of it) as P.
// A power looks up two entries, each in the middle of its dependent chain and
// each lane its own: LDS answers in half the time of the vector cache.  The
// steps' kernels therefore copy the tables to LDS (5 KiB a block), the sweeps and
// the unsplit tile while their first global loads are in flight, the 1D ensemble
// and the unsplit strip before them.  A step before and after: split 64^2 .0751
// -> .0724 ms, 1024^2 .391 -> .377, 4096^2 learned 4.86 -> 4.55; unsplit 1024^2
// .337 -> .327, learned .412 -> .381; two fluids 2048 x 512 .539 -> .512.
static constexpr int POW_TAB = powtab::EXP_BASE + 128 * powtab::EXP_ROW;
#if defined(__HIPCC__)
template <int N>
struct TabLoad {                  // the part of the tables that one of N threads copies
    static constexpr int PER = (POW_TAB + N - 1) / N;
    double v[PER];
    __device__ __forceinline__ void load(int id)
    {
#pragma unroll
        for (int k = 0; k < PER; ++k) v[k] = powtab::TAB[min(id + k * N, POW_TAB - 1)];
    }
    __device__ __forceinline__ void store(int id, double *tab) const
    {
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if (id + k * N < POW_TAB) tab[id + k * N] = v[k];
    }
};
#endif

HGRP_HD DD log_in_range(double x, const double *P)            // x positive, normal
{
    int k;
    double m = frexp(x, &k);
    m *= 2.0;
    k -= 1;
    const int j = (int)fma(m, 128.0, -128.0) & 127;
    const double *lt = P + powtab::LOG_ROW * j;
    const double invc = lt[0];
    const double r = fma(m, invc, -1.0);
    const double q_hi = r * r;
    const double q_lo = fma(r, r, -q_hi);
    double t = -1.0 / 10.0;
    t = fma(t, r, 1.0 / 9.0);
    t = fma(t, r, -1.0 / 8.0);
    t = fma(t, r, 1.0 / 7.0);
    t = fma(t, r, -1.0 / 6.0);
    t = fma(t, r, 1.0 / 5.0);
    t = fma(t, r, -1.0 / 4.0);
    t = fma(t, r, 1.0 / 3.0);
    const double tail = t * (q_hi * r);
    const double kd = (double)k;
    const DD s1 = fast_sum(kd * powtab::LN2_HI, lt[1]);   // k = 0, or |k| ln2 >= log c
    const DD s2 = two_sum(s1.hi, r);
    const DD s3 = two_sum(s2.hi, -0.5 * q_hi);
    const double lo = fma(-0.5, q_lo, s1.lo + s2.lo + s3.lo + kd * powtab::LN2_LO + lt[2]) + tail;
    const double hi = s3.hi + lo;
    return {hi, lo - (hi - s3.hi)};
}

HGRP_HD double exp_in_range(DD p, const double *P)            // |p.hi| < 700
{
    const double kf = rint(p.hi * powtab::INV_LN2N);
    const int k2 = (int)kf;
    const DD z = two_sum(fma(-kf, powtab::LN2N_HI, p.hi), p.lo - kf * powtab::LN2N_LO);   // kf LN2N_HI is exact
    const double z_hi = z.hi, z_lo = z.lo;
    double t = 1.0 / 5040.0;
    t = fma(t, z_hi, 1.0 / 720.0);
    t = fma(t, z_hi, 1.0 / 120.0);
    t = fma(t, z_hi, 1.0 / 24.0);
    t = fma(t, z_hi, 1.0 / 6.0);
    t = fma(t, z_hi, 0.5);
    const double small = z_lo + z_hi * z_lo + (z_hi * z_hi) * t;
    const double *et = P + powtab::EXP_BASE + powtab::EXP_ROW * (k2 & 127);
    const double T_hi = et[0], T_lo = et[1];
    const double prod_hi = T_hi * z_hi;
    const double prod_lo = fma(T_hi, z_hi, -prod_hi);
    const DD s = fast_sum(T_hi, prod_hi);                  // T_hi >= 1 > |prod_hi|
    const double tail = s.lo + prod_lo + T_hi * small + T_lo + T_lo * (z_hi + small);
    return ldexp(s.hi + tail, k2 >> 7);
}

// x^y from L = log(x): pow_with for x in range and |y log x| < 700
HGRP_HD double pow_in_range(const DD &L, double y, const double *P)
{
    const double p_hi = y * L.hi;
    const double p_lo = fma(y, L.hi, -p_hi) + y * L.lo;
    return exp_in_range(fast_sum(p_hi, p_lo), P);
}

}  // namespace hgrp
