// sweep2d_tf.hip -- the directional sweeps for two gamma-law fluids.
//
// Same schedule, limiter, reconstruction, GRP solve and update as sweep2d.hip,
// with a fifth cell quantity: the volume fraction a of fluid a.  It is limited
// and reconstructed like the others, carried through the GRP solver with the
// contact (grp_2d_flux_tf), and advanced in quasi-conservative form
//     a_new = a - nu ((u_n a)_r - (u_n a)_l - a ((u_n)_r - (u_n)_l))
// with u_n and a at t + tau/2 on the interfaces.  Because 1/(gamma-1) is
// linear in a and the energy flux uses the same interface values, a uniform
// pressure and velocity across a material interface stay uniform.  In cells
// with a = 1 (or 0) every operation is the single-fluid one, bit for bit.
// Boundary conditions: -2, -4, -7, -24 (the initial-value ghosts of -1 are not
// kept for a).
#include <hip/hip_runtime.h>
#include "grp_device.hpp"
#include "sweep2d.hpp"

namespace hgrp {

constexpr int NQ = 5;   // rho u v p a

template <int DIR>
struct LineTF {
    const SweepArgs &a;
    size_t base, stride;
    int cnt;
    static constexpr int NV = DIR == 0 ? 1 : 2;

    __device__ LineTF(const SweepArgs &args, int ln) : a(args)
    {
        if (DIR == 0) { base = (size_t)ln; stride = (size_t)args.ld; cnt = args.m; }
        else          { base = (size_t)ln * (size_t)args.ld; stride = 1; cnt = args.n; }
    }
    __device__ size_t at(int k) const { return base + (size_t)k * stride; }
    __device__ void cell(int k, double w[NQ]) const
    {
        const size_t o = at(k);
        const double *f = a.st + o;
        w[0] = f[0]; w[1] = f[a.plane]; w[2] = f[2 * a.plane]; w[3] = f[3 * a.plane]; w[4] = a.fa[o];
    }
    __device__ void value(int k, double w[NQ]) const
    {
        if (k >= 0 && k < cnt) { cell(k, w); return; }
        const bool lo = k < 0;
        switch (a.bc) {
        case BC_PERIODIC:
            cell(lo ? cnt - 1 : 0, w);
            return;
        case BC_REFLECT:
            cell(lo ? 0 : cnt - 1, w);
            w[NV] = -w[NV];
            return;
        case BC_REFLECT_FREE:
            cell(lo ? 0 : cnt - 1, w);
            if (lo) w[NV] = -w[NV];
            return;
        default:
            cell(lo ? 0 : cnt - 1, w);
            return;
        }
    }
    __device__ void prev_slopes(int k, double sp[NQ]) const
    {
        const size_t o = at(k);
        for (int q = 0; q < 4; ++q) sp[q] = a.limiter3 ? a.s[o + q * a.plane] : 0.0;
        sp[4] = a.limiter3 ? a.sa[o] : 0.0;
    }
    __device__ void limited_sp(const double vm[NQ], const double v0[NQ], const double vp[NQ], const double sp[NQ],
                               double s[NQ]) const
    {
        double d_L[NQ], d_R[NQ], s_L[NQ], s_R[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) { d_L[q] = v0[q] - vm[q]; d_R[q] = vp[q] - v0[q]; }
        quot4<NQ>(d_L, a.div_h, s_L);
        quot4<NQ>(d_R, a.div_h, s_R);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            s[q] = a.limiter3 ? minmod3(a.alpha * s_L[q], a.alpha * s_R[q], sp[q]) : minmod2(s_L[q], s_R[q]);
    }
    __device__ void limited_at(int k, double s[NQ]) const
    {
        double vm[NQ], v0[NQ], vp[NQ], sp[NQ];
        value(k - 1, vm); value(k, v0); value(k + 1, vp);
        prev_slopes(k, sp);
        limited_sp(vm, v0, vp, sp, s);
    }
    // ghost slopes as in sweep2d.hip; the volume fraction is a scalar like rho
    __device__ void ghost_slope(bool lo, double s[NQ]) const
    {
        for (int q = 0; q < NQ; ++q) s[q] = 0.0;
        double t[NQ];
        switch (a.bc) {
        case BC_REFLECT:
            limited_at(lo ? 0 : cnt - 1, t);
            s[NV] = t[NV];
            break;
        case BC_PERIODIC:
            limited_at(lo ? cnt - 1 : 0, s);
            break;
        case BC_REFLECT_FREE:
            if (lo) { limited_at(0, t); s[NV] = t[NV]; }
            break;
        default:
            break;
        }
    }
    // ghost slopes next to a boundary cell whose own slopes `near` the caller has: the rules of
    // ghost_slope, which only the periodic one needs other cells for
    __device__ void ghost_slope_near(bool lo, const double near[NQ], double s[NQ]) const
    {
        if (a.bc == BC_PERIODIC) {
            limited_at(lo ? cnt - 1 : 0, s);
            return;
        }
        const bool keep = a.bc == BC_REFLECT || (a.bc == BC_REFLECT_FREE && lo);
#pragma unroll
        for (int q = 0; q < NQ; ++q) s[q] = keep && q == NV ? near[q] : 0.0;
    }
    // update of cell k: the single-fluid update with the mixture's gamma, and
    // the volume fraction in quasi-conservative form
    __device__ void update(int k, const double w[NQ], double e, const double Fl[4], const double Fr[4],
                           const double Zl[3], const double Zr[3], const double Il[4], const double Ir[4]) const
    {
        const size_t o = at(k);
        const double nu = a.nu;
        const double mom_x = w[0] * w[1] - nu * (Fr[1] - Fl[1]);
        const double mom_y = w[0] * w[2] - nu * (Fr[2] - Fl[2]);
        const double ene = w[0] * e - nu * (Fr[3] - Fl[3]);
        const double rho = w[0] + -nu * (Fr[0] - Fl[0]);
        double u, v, e_new;
        quot3(mom_x, mom_y, ene, rho, u, v, e_new);
        double fa = w[4] - nu * ((Zr[0] - Zl[0]) - w[4] * (Zr[1] - Zl[1]));
        fa = fmin(fmax(fa, 0.0), 1.0);
        const double X = ene - 0.5 * mom_x * u - 0.5 * mom_y * v;
        double p;
        if (fa == 1.0) p = X * a.two.a.gm1();
        else if (fa == 0.0) p = X * a.two.b.gm1();
        else if (two_in_range(a.two) && fabs(X) >= 0x1p-300 && fabs(X) <= 0x1p300) p = div_1(X, mix_inv_gm1_q(fa, a.two));
        else p = X / (fa / (a.two.a.g - 1.0) + (1.0 - fa) / (a.two.b.g - 1.0));
        double *f = a.st_o + o;
        const size_t P = a.plane;
        f[0] = rho; f[P] = u; f[2 * P] = v; f[4 * P] = e_new; f[3 * P] = p; a.fa_o[o] = fa;
        if (p < a.eps || rho < a.eps) atomicOr(&a.status->flags, 1u);
        const double dI[NQ] = {Ir[0] - Il[0], Ir[1] - Il[1], Ir[2] - Il[2], Ir[3] - Il[3], Zr[2] - Zl[2]};
        double sn[NQ];
        quot4<NQ>(dI, a.div_h, sn);
#pragma unroll
        for (int q = 0; q < 4; ++q) a.s_o[o + q * P] = sn[q];
        a.sa_o[o] = sn[4];
    }
};

__device__ __forceinline__ void recon_tf(const double w[NQ], const double s[NQ], double hh, bool left, Side &f,
                                         double &fa, double &d_fa)
{
    if (left) {
        f.rho = w[0] + hh * s[0]; f.u = w[1] + hh * s[1]; f.v = w[2] + hh * s[2]; f.p = w[3] + hh * s[3];
        fa = w[4] + hh * s[4];
    } else {
        f.rho = w[0] - hh * s[0]; f.u = w[1] - hh * s[1]; f.v = w[2] - hh * s[2]; f.p = w[3] - hh * s[3];
        fa = w[4] - hh * s[4];
    }
    f.d_rho = s[0]; f.d_u = s[1]; f.d_v = s[2]; f.d_p = s[3];
    d_fa = s[4];
}

// Face f of grid line `line` (between cells f - 1 and f) with the IEEE solver,
// from the cells in memory: what the fast solver leaves (grp_fast.hpp).
// FIZ: flux, values at t + tau, the fraction's three.
template <int DIR, bool CONV>
__device__ __attribute__((noinline)) int redo_face_tf(const SweepArgs *ap, int line, int f, double p_guess, double *FIZ)
{
    const SweepArgs &a = *ap;
    const LineTF<DIR> L(a, line);
    double wl[NQ], wr[NQ], sl[NQ], sr[NQ], FA[4];
    L.value(f - 1, wl);
    L.value(f, wr);
    if (f > 0) L.limited_at(f - 1, sl); else L.ghost_slope(true, sl);
    if (f < L.cnt) L.limited_at(f, sr); else L.ghost_slope(false, sr);
    Side SL, SR;
    recon_tf(wl, sl, a.hh, true, SL, FA[0], FA[1]);
    recon_tf(wr, sr, a.hh, false, SR, FA[2], FA[3]);
    return grp_2d_flux_tf<DIR, CONV>(SL, SR, a.two, FA, a.tau, a.eps, FIZ, FIZ + 4, FIZ + 8, a.tol, p_guess);
}

template <int DIR, int NM>
__device__ __forceinline__ void solve_interface_tf(const SweepArgs &a, const double wl[NQ], const double sl[NQ],
                                                   const double wr[NQ], const double sr[NQ], int line, int f, double F[4],
                                                   double I[4], double Z[3], const double *tab, double p_guess = -1.0)
{
    Side SL, SR;
    double FA[4];
    recon_tf(wl, sl, a.hh, true, SL, FA[0], FA[1]);
    recon_tf(wr, sr, a.hh, false, SR, FA[2], FA[3]);
    int code = ifvar_bad(SL, SR, a.eps) ? 1 : 0, bad = 0;
    const bool done = flux_two_fluid_q<DIR, NM != NM_REF>(SL, SR, a.two, FA, a.near2, a.tau, a.eps, F, I, Z, a.tol,
                                                          p_guess, &bad, tab);
    if (__builtin_expect(__any(!done), 0)) {
        if (!done) {
            const SweepArgs ar = reload_args<SweepArgs>();
            double o[11];
            bad = redo_face_tf<DIR, NM != NM_REF>(&ar, line, f, p_guess, o);
#pragma unroll
            for (int q = 0; q < 4; ++q) { F[q] = o[q]; I[q] = o[4 + q]; }
#pragma unroll
            for (int q = 0; q < 3; ++q) Z[q] = o[8 + q];
        }
    }
    if (bad) code = 2;
    if (code) {
        const SweepArgs ar = reload_args<SweepArgs>();
        const unsigned long long index = (unsigned long long)line * (unsigned long long)((DIR == 0 ? ar.m : ar.n) + 1)
                                         + (unsigned long long)f;
        atomicMax(&ar.status->fail_key, ((index << 2) | (unsigned long long)code) + 1ull);
    }
}

// learned starting pressure for the interface (wl, sl | wr, sr), every lane of
// the wave (uniform call); gamma of each side from its reconstructed fraction
template <int DIR>
__device__ __forceinline__ double interface_guess_tf(const SweepArgs &a, bool active, const double wl[NQ],
                                                     const double sl[NQ], const double wr[NQ], const double sr[NQ],
                                                     uint32_t *lds)
{
    Side SL, SR;
    double aL, daL, aR, daR;
    recon_tf(wl, sl, a.hh, true, SL, aL, daL);
    recon_tf(wr, sr, a.hh, false, SR, aR, daR);
    const double uL = DIR == 0 ? SL.u : SL.v, uR = DIR == 0 ? SR.u : SR.v;
    const double dist2 = (SL.rho - SR.rho) * (SL.rho - SR.rho) + (uL - uR) * (uL - uR) + (SL.p - SR.p) * (SL.p - SR.p);
    // Newton runs only past the acoustic shortcut and the equal-state exit of the exact solver
    const bool want = active && !(dist2 < a.near2) && !(fabs(uL - uR) < a.tol && fabs(SL.p - SR.p) < a.tol);
    const double gL = aL == 1.0 ? a.two.a.g : (aL == 0.0 ? a.two.b.g : mix_gamma_q(aL, a.two));
    const double gR = aR == 1.0 ? a.two.a.g : (aR == 0.0 ? a.two.b.g : mix_gamma_q(aR, a.two));
    return learned_guess_wave(a.mlp, want, SL.rho, uL, SL.p, SR.rho, uR, SR.p, gL, gR, lds);
}

__device__ __forceinline__ bool tf_halted(const SweepArgs &a)
{
    if (a.prev == nullptr) return false;
    const SweepStatus pv = *a.prev;
    if (pv.fail_key != 0ull || pv.flags != 0u) {
        if (threadIdx.x == 0) atomicOr(&a.status->flags, 2u);
        return true;
    }
    return false;
}

// Both sweeps in the wave form of the single-fluid ones (wave_sweep), lines of 16
// cells (X of few cells: x_lanes), a register budget for three waves per SIMD (33-36
// registers spilled; a step of 2048 x 512 with the learned guess .403 ms, at two
// waves .473, at four .614; converge rule .434, .502 and .528).
template <int DIR, int NM, int G>
__device__ __forceinline__ void wave_sweep_tf(const SweepArgs &a, int per_row, double (*st)[64], uint32_t *mlp, double *tab)
{
    constexpr bool LEARNED = NM == NM_LEARNED;
    constexpr int LINES = 64 / G, STEP = DIR == 0 ? LINES : 1;   // STEP: lanes between neighbours along the sweep
    const int lane = threadIdx.x & 63, k = DIR == 0 ? lane / LINES : lane % G;
    const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int slow = (int)(wave / per_row), fast = (int)(wave % per_row);
    const int j = (DIR == 0 ? fast : slow) * LINES + (DIR == 0 ? lane % LINES : lane / G);
    const bool rowv = j < (DIR == 0 ? a.n : a.m);
    const int c0 = (DIR == 0 ? slow : fast) * (G - 1);
    const int n = DIR == 0 ? a.m : a.n;                          // cells along the sweep
    const int c = c0 - 1 + k;
    const LineTF<DIR> L(a, rowv ? j : 0);

    const bool own = rowv && c >= 0 && c < n;
    double w[NQ] = {1.0, 0.0, 0.0, 1.0, 1.0}, sp[NQ] = {0.0, 0.0, 0.0, 0.0, 0.0}, e_c = 0.0;
    if (rowv && c <= n) L.value(c, w);
    if (own) {
        L.prev_slopes(c, sp);
        e_c = a.st[L.at(c) + 4 * a.plane];
    }
    const bool first = rowv && k == 0 && c >= 0, last = rowv && k == G - 1 && c + 1 <= n;
    const bool last_own = rowv && k == G - 1 && c + 1 < n;
    double wl_e[NQ], wr_e[NQ], wrr[NQ], sp1[NQ];
    if (first) L.value(c - 1, wl_e);
    if (last) L.value(c + 1, wr_e);
    if (last_own) {
        L.value(c + 2, wrr);
        L.prev_slopes(c + 1, sp1);
    }
    TabLoad<256> tl;
    tl.load(threadIdx.x);
    // the predecessor's status is read while the loads above are in flight; the
    // whole block returns together
    if (tf_halted(a)) return;
    tl.store(threadIdx.x, tab);
    __syncthreads();
    if (!__any(rowv) || c0 >= n) return;                         // a wave past the last line or cell
#pragma unroll
    for (int q = 0; q < NQ; ++q) st[q][lane] = w[q];
    st[NQ][lane] = e_c;
    double wl[NQ], wr[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) { wl[q] = __shfl_up(w[q], STEP); wr[q] = __shfl_down(w[q], STEP); }
    if (first)
#pragma unroll
        for (int q = 0; q < NQ; ++q) wl[q] = wl_e[q];
    if (last)
#pragma unroll
        for (int q = 0; q < NQ; ++q) wr[q] = wr_e[q];

    double s[NQ] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (own) L.limited_sp(wl, w, wr, sp, s);
    double sr[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) sr[q] = __shfl_down(s[q], STEP);
    if (last_own) L.limited_sp(w, wr, wrr, sp1, sr);
    // the ghosts' slopes from the boundary cells'
    if (rowv && (c == -1 || c + 1 == n)) {
        double g[NQ];
        L.ghost_slope_near(c == -1, c == -1 ? sr : s, g);
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (c == -1) s[q] = g[q]; else sr[q] = g[q];
        }
    }

    double F[4] = {0.0, 0.0, 0.0, 0.0}, I[4] = {0.0, 0.0, 0.0, 0.0}, Z[3] = {0.0, 0.0, 0.0};
    const int f = c + 1;
    const bool face = rowv && f <= n;
    double pg = -1.0;
    if constexpr (LEARNED) pg = interface_guess_tf<DIR>(a, face, w, s, wr, sr, mlp);
    if (face)
        solve_interface_tf<DIR, NM>(a, w, s, wr, sr, j, f, F, I, Z, tab, pg);
    double Fl[4], Il[4], Zl[3];
#pragma unroll
    for (int q = 0; q < 4; ++q) { Fl[q] = __shfl_up(F[q], STEP); Il[q] = __shfl_up(I[q], STEP); }
#pragma unroll
    for (int q = 0; q < 3; ++q) Zl[q] = __shfl_up(Z[q], STEP);
    if (k >= 1 && own) {
        double wc[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q) wc[q] = st[q][lane];
        const SweepArgs ar = reload_args<SweepArgs>();   // not held across the solve
        LineTF<DIR>(ar, j).update(c, wc, st[NQ][lane], Fl, F, Zl, Z, Il, I);
    }
}

template <int NM, int G>
__global__ void __launch_bounds__(256, 3) sweep_x_tf_kernel(SweepArgs a, int per_row)
{
    constexpr bool LEARNED = NM == NM_LEARNED;
    __shared__ double stash[4][NQ + 1][64];
    __shared__ uint32_t mlp_lds[LEARNED ? 4 : 1][LEARNED ? 64 * 8 : 1];
    __shared__ double tab[POW_TAB];
    const int wv = (threadIdx.x >> 6) & 3;
    wave_sweep_tf<0, NM, G>(a, per_row, stash[wv], mlp_lds[wv], tab);
}

template <int NM, int G>
__global__ void __launch_bounds__(256, 3) sweep_y_tf_kernel(SweepArgs a, int per_row)
{
    constexpr bool LEARNED = NM == NM_LEARNED;
    __shared__ double stash[4][NQ + 1][64];
    __shared__ uint32_t mlp_lds[LEARNED ? 4 : 1][LEARNED ? 64 * 8 : 1];
    __shared__ double tab[POW_TAB];
    const int wv = (threadIdx.x >> 6) & 3;
    wave_sweep_tf<1, NM, G>(a, per_row, stash[wv], mlp_lds[wv], tab);
}

// min over cells of min(h_x, h_y) / (|c| + |u| + |v|) with the mixture's gamma
__global__ void __launch_bounds__(256) cfl_tf_kernel(const double *rho, const double *u, const double *v,
                                                     const double *p, const double *fa, int m, int n, int ld,
                                                     TwoGas two, double hmin, unsigned long long *out)
{
    double best = INFINITY;
    const long total = (long)m * n;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (long)gridDim.x * blockDim.x) {
        const long jj = k / n, ii = k % n;
        const size_t o = (size_t)jj * ld + ii;
        const double g = gas_of(fa[o], two).g;
        const double c = sqrt(g * p[o] / rho[o]);
        const double sigma = fabs(c) + fabs(u[o]) + fabs(v[o]);
        best = fmin(best, hmin / sigma);
    }
    for (int off = 32; off > 0; off >>= 1) best = fmin(best, __shfl_xor(best, off));
    if ((threadIdx.x & 63) == 0) {
        unsigned long long bits = __double_as_longlong(best);
        if (!(best >= 0.0)) bits = 0x7ff0000000000000ull;
        atomicMin(out, bits);
    }
}

// E of every cell from its primitives with the mixture's gamma: the reference
// main program's expression (src/hydrocode_2D/hydrocode.c:251-252) in pure
// cells, and p * (a/(gamma_a-1) + (1-a)/(gamma_b-1)) / rho in mixed ones, the
// exact inverse of the pressure the update forms there.
__global__ void __launch_bounds__(256) energy_tf_kernel(const double *rho, const double *u, const double *v,
                                                        const double *p, const double *fa, double *e, int m, int n,
                                                        int ld, TwoGas two)
{
    const long total = (long)m * n;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (long)gridDim.x * blockDim.x) {
        const long jj = k / n, ii = k % n;
        const size_t o = (size_t)jj * ld + ii;
        const double a = fa[o];
        double E;
        if (a == 1.0 || a == 0.0) {
            const double g = a == 1.0 ? two.a.g : two.b.g;
            E = 0.5 * u[o] * u[o] + p[o] / (g - 1.0) / rho[o];
        } else {
            E = 0.5 * u[o] * u[o] + p[o] * (a / (two.a.g - 1.0) + (1.0 - a) / (two.b.g - 1.0)) / rho[o];
        }
        e[o] = E + 0.5 * v[o] * v[o];
    }
}

hipError_t launch_energy_tf(const double *rho, const double *u, const double *v, const double *p, const double *fa,
                            double *e, int m, int n, int ld, const TwoGas &two, hipStream_t st)
{
    const long total = (long)m * n;
    long blocks = (total + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(energy_tf_kernel, dim3((unsigned)blocks), dim3(256), 0, st, rho, u, v, p, fa, e, m, n, ld, two);
    return hipGetLastError();
}

static int x_tf_lanes(int m, int n)
{
    return x_lanes(wave_grid(0, m, n, 16).blocks, wave_grid(0, m, n, 8).blocks, wave_grid(0, m, n, 4).blocks);
}

// the two-fluid sweep kernel's name as profilers print it
const char *sweep_tf_kernel_name(int dir, int nm, int m, int n)
{
    static const char *xn[3][3] = {
        {"sweep_x_tf_kernel<0, 16>", "sweep_x_tf_kernel<1, 16>", "sweep_x_tf_kernel<2, 16>"},
        {"sweep_x_tf_kernel<0, 8>", "sweep_x_tf_kernel<1, 8>", "sweep_x_tf_kernel<2, 8>"},
        {"sweep_x_tf_kernel<0, 4>", "sweep_x_tf_kernel<1, 4>", "sweep_x_tf_kernel<2, 4>"}};
    static const char *yn[3] = {"sweep_y_tf_kernel<0, 16>", "sweep_y_tf_kernel<1, 16>", "sweep_y_tf_kernel<2, 16>"};
    if (nm < 0 || nm > 2 || dir < 0 || dir > 1) return "";
    const int G = x_tf_lanes(m, n);
    return dir == 0 ? xn[G == 16 ? 0 : G == 8 ? 1 : 2][nm] : yn[nm];
}

template <int G>
static hipError_t launch_x_tf(const SweepArgs &a, hipStream_t st)
{
    const WaveGrid w = wave_grid(0, a.m, a.n, G);
    const dim3 grid((unsigned)w.blocks), block(256);
    switch (newton_mode(a)) {
    case NM_LEARNED: hipLaunchKernelGGL((sweep_x_tf_kernel<NM_LEARNED, G>), grid, block, 0, st, a, w.per_row); break;
    case NM_CONV: hipLaunchKernelGGL((sweep_x_tf_kernel<NM_CONV, G>), grid, block, 0, st, a, w.per_row); break;
    default: hipLaunchKernelGGL((sweep_x_tf_kernel<NM_REF, G>), grid, block, 0, st, a, w.per_row); break;
    }
    return hipGetLastError();
}

hipError_t launch_sweep_x_tf(const SweepArgs &a, hipStream_t st)
{
    switch (x_tf_lanes(a.m, a.n)) {
    case 4: return launch_x_tf<4>(a, st);
    case 8: return launch_x_tf<8>(a, st);
    default: return launch_x_tf<16>(a, st);
    }
}

hipError_t launch_sweep_y_tf(const SweepArgs &a, hipStream_t st)
{
    const WaveGrid w = wave_grid(1, a.m, a.n, 16);
    const dim3 grid((unsigned)w.blocks), block(256);
    switch (newton_mode(a)) {
    case NM_LEARNED: hipLaunchKernelGGL((sweep_y_tf_kernel<NM_LEARNED, 16>), grid, block, 0, st, a, w.per_row); break;
    case NM_CONV: hipLaunchKernelGGL((sweep_y_tf_kernel<NM_CONV, 16>), grid, block, 0, st, a, w.per_row); break;
    default: hipLaunchKernelGGL((sweep_y_tf_kernel<NM_REF, 16>), grid, block, 0, st, a, w.per_row); break;
    }
    return hipGetLastError();
}

hipError_t launch_cfl_tf(const double *rho, const double *u, const double *v, const double *p, const double *fa,
                         int m, int n, int ld, const TwoGas &two, double hmin, unsigned long long *out, hipStream_t st)
{
    const long total = (long)m * n;
    long blocks = (total + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(cfl_tf_kernel, dim3((unsigned)blocks), dim3(256), 0, st, rho, u, v, p, fa, m, n, ld, two, hmin,
                       out);
    return hipGetLastError();
}

}  // namespace hgrp
