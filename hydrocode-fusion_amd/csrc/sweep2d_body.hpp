// sweep2d_body.hpp -- the bodies of the directional sweeps of the
// dimension-split 2D GRP step, shared by the one-grid kernels (sweep2d.hip)
// and the kernels that advance a batch of grids (grp2d_batch.hip).
//
// Semantics follow src/finite_volume/grp_solver_2D_split_EUL_source.c:182-303,
// src/inter_process/bound_cond_slope_limiter_{x,y}.c:27-129,
// src/inter_process/slope_limiter{,_2D_x}.c and src/flux_calc/flux_generator_{x,y}.c:31-165.
#pragma once
#include <hip/hip_runtime.h>

#include "grp_device.hpp"
#include "sweep2d.hpp"

namespace hgrp {

// The argument block of a one-grid sweep kernel, read again from
// kernel-argument memory (see reload_args).
struct KernargArgs {
    __device__ SweepArgs get() const { return reload_args<SweepArgs>(); }
};

__device__ __forceinline__ bool sweep_halted(const SweepArgs &a)
{
    if (a.prev == nullptr) return false;
    const SweepStatus pv = *a.prev;
    if (pv.fail_key != 0ull || pv.flags != 0u) {
        if (threadIdx.x == 0) atomicOr(&a.status->flags, 2u);
        return true;
    }
    return false;
}

// One grid line along the sweep direction.  DIR 0: x-line i (cells j = 0..m-1,
// stride ld); DIR 1: y-line j (cells i = 0..n-1, stride 1).  Index -1 and cnt
// are the ghost cells.
template <int DIR>
struct Line {
    const SweepArgs &a;
    size_t base, stride;
    int cnt, line;
    static constexpr int NV = DIR == 0 ? 1 : 2;   // normal velocity: u in x, v in y

    __device__ Line(const SweepArgs &args, int ln) : a(args), line(ln)
    {
        if (DIR == 0) { base = (size_t)ln; stride = (size_t)args.ld; cnt = args.m; }
        else          { base = (size_t)ln * (size_t)args.ld; stride = 1; cnt = args.n; }
    }
    __device__ size_t at(int k) const { return base + (size_t)k * stride; }

    __device__ void cell(int k, double w[4]) const
    {
        const size_t o = at(k);
        const double *f = a.st + o;
        w[0] = f[0]; w[1] = f[a.plane]; w[2] = f[2 * a.plane]; w[3] = f[3 * a.plane];
    }
    // value of cell k, ghost values at k == -1 / k == cnt (bound_cond_slope_limiter_x.c:34-82)
    __device__ void value(int k, double w[4]) const
    {
        if (k >= 0 && k < cnt) { cell(k, w); return; }
        const bool lo = k < 0;
        switch (a.bc) {
        case BC_INITIAL: {
            const double *b = (lo ? a.bnd_lo : a.bnd_hi) + (size_t)line * 4;
            w[0] = b[0]; w[1] = b[1]; w[2] = b[2]; w[3] = b[3];
            return;
        }
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
        default:   // BC_FREE
            cell(lo ? 0 : cnt - 1, w);
            return;
        }
    }
    // previous slopes of cell k (read by minmod3 only)
    __device__ void prev_slopes(int k, double sp[4]) const
    {
        const size_t o = at(k);
#pragma unroll
        for (int q = 0; q < 4; ++q) sp[q] = a.limiter3 ? a.s[o + q * a.plane] : 0.0;
    }
    // limited slope from the neighbours and the previous slope sp (slope_limiter_2D_x.c:177-211)
    __device__ void limited_sp(const double vm[4], const double v0[4], const double vp[4], const double sp[4],
                               double s[4]) const
    {
        double d_L[4], d_R[4], s_L[4], s_R[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) { d_L[q] = v0[q] - vm[q]; d_R[q] = vp[q] - v0[q]; }
        quot4(d_L, a.div_h, s_L);
        quot4(d_R, a.div_h, s_R);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            s[q] = a.limiter3 ? minmod3(a.alpha * s_L[q], a.alpha * s_R[q], sp[q]) : minmod2(s_L[q], s_R[q]);
    }
    __device__ void limited(int k, const double vm[4], const double v0[4], const double vp[4], double s[4]) const
    {
        double sp[4];
        prev_slopes(k, sp);
        limited_sp(vm, v0, vp, sp, s);
    }
    __device__ void limited_at(int k, double s[4]) const
    {
        double vm[4], v0[4], vp[4];
        value(k - 1, vm); value(k, v0); value(k + 1, vp);
        limited(k, vm, v0, vp, s);
    }
    // ghost slopes (bound_cond_slope_limiter_x.c:94-109); zero where the reference leaves them unset
    __device__ void ghost_slope(bool lo, double s[4]) const
    {
        s[0] = s[1] = s[2] = s[3] = 0.0;
        double t[4];
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
    __device__ void ghost_slope_near(bool lo, const double near[4], double s[4]) const
    {
        if (a.bc == BC_PERIODIC) {
            limited_at(lo ? cnt - 1 : 0, s);
            return;
        }
        const bool keep = a.bc == BC_REFLECT || (a.bc == BC_REFLECT_FREE && lo);
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = keep && q == NV ? near[q] : 0.0;
    }
    // conservative update of cell k (e: its E) and slope refresh (grp_solver_2D_split_EUL_source.c:236-254)
    __device__ void update(int k, const double w[4], const double e, const double Fl[4], const double Fr[4],
                           const double Il[4], const double Ir[4]) const
    {
        const size_t o = at(k);
        const double nu = a.nu;
        const double mom_x = w[0] * w[1] - nu * (Fr[1] - Fl[1]);
        const double mom_y = w[0] * w[2] - nu * (Fr[2] - Fl[2]);
        const double ene = w[0] * e - nu * (Fr[3] - Fl[3]);
        const double rho = w[0] + -nu * (Fr[0] - Fl[0]);
        double u, v, e_new;
        quot3(mom_x, mom_y, ene, rho, u, v, e_new);
        const double p = (ene - 0.5 * mom_x * u - 0.5 * mom_y * v) * a.gas.gm1();
        double *f = a.st_o + o;
        const size_t P = a.plane;
        f[0] = rho; f[P] = u; f[2 * P] = v; f[4 * P] = e_new; f[3 * P] = p;
        if (p < a.eps || rho < a.eps) atomicOr(&a.status->flags, 1u);
        double dI[4], sn[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) dI[q] = Ir[q] - Il[q];
        quot4(dI, a.div_h, sn);
#pragma unroll
        for (int q = 0; q < 4; ++q) a.s_o[o + q * P] = sn[q];
    }
};

// Face f of grid line `line` (between cells f - 1 and f) with the IEEE solver,
// from the cells in memory: what the fast solver leaves (grp_fast.hpp).  F, I:
// the flux and the values at t + tau; returns grp_2d_flux's code.  MINW: the
// calling kernels' register budget (waves per SIMD); a copy of its own for each
// keeps the compiler from giving the callee a larger one.
template <int DIR, bool CONV, int MINW>
__device__ __attribute__((noinline)) int redo_face(const SweepArgs *ap, int line, int f, double p_guess, double *FI)
{
    const SweepArgs &a = *ap;
    const Line<DIR> L(a, line);
    double wl[4], wr[4], sl[4], sr[4];
    L.value(f - 1, wl);
    L.value(f, wr);
    if (f > 0) L.limited_at(f - 1, sl); else L.ghost_slope(true, sl);
    if (f < L.cnt) L.limited_at(f, sr); else L.ghost_slope(false, sr);
    return grp_2d_flux<DIR, CONV>(recon(wl, sl, a.hh, true), recon(wr, sr, a.hh, false), a.gas, a.tau, a.eps, FI,
                                  FI + 4, a.tol, p_guess);
}

// GRP flux of face f of grid line `line`, sides SL | SR.  src gives the
// argument block again (see reload_args).
template <int DIR, int NM, int MINW, class Src>
__device__ __forceinline__ void solve_interface(const SweepArgs &a, const Src &src, const Side &SL, const Side &SR,
                                                int line, int f, double F[4], double I[4], const double *tab,
                                                double p_guess = -1.0)
{
    int code = ifvar_bad(SL, SR, a.eps) ? 1 : 0, bad = 0;
    const bool done = flux_split_q<DIR, NM != NM_REF>(SL, SR, a.gas, a.near2, a.tau, a.eps, F, I, a.tol, p_guess, &bad,
                                                   tab);
    if (__builtin_expect(__any(!done), 0)) {
        if (!done) {
            const SweepArgs ar = src.get();
            double o[8];
            bad = redo_face<DIR, NM != NM_REF, MINW>(&ar, line, f, p_guess, o);
#pragma unroll
            for (int q = 0; q < 4; ++q) { F[q] = o[q]; I[q] = o[4 + q]; }
        }
    }
    if (bad) code = 2;
    if (code) {
        const SweepArgs ar = src.get();
        const unsigned long long index = (unsigned long long)line * (unsigned long long)((DIR == 0 ? ar.m : ar.n) + 1)
                                         + (unsigned long long)f;
        atomicMax(&ar.status->fail_key, ((index << 2) | (unsigned long long)code) + 1ull);
    }
}

// Learned starting pressure for the interface (SL | SR) normal to DIR, for
// every lane of the wave (uniform call); -1 where Newton will not run (the
// Q1D acoustic shortcut dist < eps, the solver's equal-state exit) or the lane
// has no interface.
template <int DIR>
__device__ __forceinline__ double interface_guess(const SweepArgs &a, bool active, const Side &SL, const Side &SR,
                                                  uint32_t *lds)
{
    const double uL = DIR == 0 ? SL.u : SL.v, uR = DIR == 0 ? SR.u : SR.v;
    const double dist2 = (SL.rho - SR.rho) * (SL.rho - SR.rho) + (uL - uR) * (uL - uR) + (SL.p - SR.p) * (SL.p - SR.p);
    // Newton runs only past the acoustic shortcut and the equal-state exit of the exact solver
    const bool want = active && !(dist2 < a.near2) && !(fabs(uL - uR) < a.tol && fabs(SL.p - SR.p) < a.tol);
    return learned_guess_wave(a.mlp, want, SL.rho, uL, SL.p, SR.rho, uR, SR.p, a.gas.g, a.gas.g, lds);
}

// Launch variants: lanes along a line and the register budget (waves per SIMD).
// Four waves are faster than three once a grid gives every SIMD more than three
// (an X sweep of 1024^2 .123 ms against .131, of 4096^2 with the learned guess 1.29
// against 1.42); below that the budget of three is (a step of 127 x 329 .073 ms
// with both sweeps' against .075), so that is a smaller grid's default.
// G = 16: the repeated face is 1 in 16 and a front along the lines still meets few
// waves.  An X sweep with 32, 16 and 8 lanes to a line: 1024^2 .122, .123 and .135
// ms, 4096^2 learned 1.53 (it reads the lines in 16-byte pieces), 1.29 and 1.30; a
// Y sweep with 64, 32, 16 and 8: 1024^2 .129, .122, .120 and .122 ms, 4096^2 1.26,
// 1.24, 1.21 and 1.30.  The others are the tuner's: which is fastest depends on how
// a state's fronts lie (Y of 384^2, the same kind of state: .035 with 32, .039 with
// 16).  Lines of 4 and 8 are also the default where they leave fewer lanes idle
// (x_lanes).
struct SweepShape {
    int G, minw;
};
inline SweepShape sweep_shape(int dir, int variant)
{
    static const SweepShape x[6] = {{16, 4}, {32, 4}, {8, 4}, {16, 3}, {4, 4}, {32, 3}};
    static const SweepShape y[5] = {{16, 4}, {32, 4}, {64, 4}, {8, 4}, {16, 3}};
    return dir == 0 ? x[variant] : y[variant];
}
inline int default_variant(int dir, int m, int n)
{
    const long b16 = wave_grid(dir, m, n, 16).blocks;
    const int G = dir == 0 ? x_lanes(b16, wave_grid(0, m, n, 8).blocks, wave_grid(0, m, n, 4).blocks) : 16;
    if (G < 16) return G == 8 ? 2 : 4;
    return b16 > FEW_BLOCKS ? 0 : dir == 0 ? 3 : 4;
}

// Wave-parallel sweep along DIR: a wave holds 64/G grid lines of G lanes each;
// the lane at place k of a line owns cell c0-1+k, computes interface c0+k and
// updates cell c0-1+k for k >= 1 (G-1 cells per line).  Neighbours are lanes of
// the same wave, so no wave waits for another once the pow tables are there: a
// row of waves that hands its faces on through LDS waits 40 % of the time at
// its three barriers (X of 4096^2, an earlier interface solve in both: 1.56
// ms against 1.36 with the learned guess, 1.83 against 1.50 without).
// DIR 1: the lanes of a line are consecutive (and so are its cells in memory);
// DIR 0: the lines are (lane k 64/G + l: line l, so 64/G consecutive i), and a
// block's waves take neighbouring lines, so that together they read whole cache
// lines.  Stacked lines let a front that lies along them meet few waves, each
// with many lanes on it.
// wave: the wave's index in the grid's sweep, per_row as wave_grid's; st, mlp:
// this wave's LDS slots; tab: the block's, for the pow tables; src gives the
// argument block again after the solve.
template <int DIR, int MINW, int NM, int G, class Src>
__device__ __forceinline__ void wave_sweep(const SweepArgs &a, const Src &src, long wave, int per_row,
                                           double (*st)[64], uint32_t *mlp, double *tab)
{
    static_assert(G == 64 || G == 32 || G == 16 || G == 8 || G == 4, "lanes per line");
    constexpr int LINES = 64 / G, STEP = DIR == 0 ? LINES : 1;   // STEP: lanes between neighbours along the sweep
    constexpr bool LEARNED = NM == NM_LEARNED;
    const int lane = threadIdx.x & 63, k = DIR == 0 ? lane / LINES : lane % G;
    const int slow = (int)(wave / per_row), fast = (int)(wave % per_row);
    const int j = (DIR == 0 ? fast : slow) * LINES + (DIR == 0 ? lane % LINES : lane / G);
    const bool rowv = j < (DIR == 0 ? a.n : a.m);
    const int c0 = (DIR == 0 ? slow : fast) * (G - 1);
    const int n = DIR == 0 ? a.m : a.n;                // cells along the sweep
    const int c = c0 - 1 + k;
    const Line<DIR> L(a, rowv ? j : 0);
    const double hh = a.hh;

    const bool own = rowv && c >= 0 && c < n;
    // every global load of the wave up front, so that it pays one memory
    // latency: the owned cell (values, previous slopes, E); the first lane of a
    // row also the cell below it; the last lane the two cells above it and the
    // previous slopes of the first (it limits that cell, the right side of its
    // interface)
    double w[4] = {1.0, 0.0, 0.0, 1.0}, sp[4] = {0.0, 0.0, 0.0, 0.0}, e_c = 0.0;
    if (rowv && c <= n) L.value(c, w);
    if (own) {
        L.prev_slopes(c, sp);
        e_c = a.st[L.at(c) + 4 * a.plane];
    }
    const bool first = rowv && k == 0 && c >= 0, last = rowv && k == G - 1 && c + 1 <= n;
    const bool last_own = rowv && k == G - 1 && c + 1 < n;
    double wl_e[4], wr_e[4], wrr[4], sp1[4];
    if (first) L.value(c - 1, wl_e);
    if (last) L.value(c + 1, wr_e);
    if (last_own) {
        L.value(c + 2, wrr);
        L.prev_slopes(c + 1, sp1);
    }
    TabLoad<256> t;
    t.load(threadIdx.x);
    // the predecessor's status is read while the loads above are in flight; the
    // whole block returns together
    if (sweep_halted(a)) return;
    t.store(threadIdx.x, tab);
    __syncthreads();
    if (!__any(rowv) || c0 >= n) return;               // a wave past the last line or cell
    // each lane reads back only its own slots: no barrier needed
#pragma unroll
    for (int q = 0; q < 4; ++q) st[q][lane] = w[q];
    st[4][lane] = e_c;
    // neighbours along the row from the next lanes; a row's end lanes take the loaded ones
    double wl[4], wr[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) { wl[q] = __shfl_up(w[q], STEP); wr[q] = __shfl_down(w[q], STEP); }
    if (first)
#pragma unroll
        for (int q = 0; q < 4; ++q) wl[q] = wl_e[q];
    if (last)
#pragma unroll
        for (int q = 0; q < 4; ++q) wr[q] = wr_e[q];

    double s[4] = {0.0, 0.0, 0.0, 0.0};
    if (own) L.limited_sp(wl, w, wr, sp, s);

    double sr[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) sr[q] = __shfl_down(s[q], STEP);
    if (last_own) L.limited_sp(w, wr, wrr, sp1, sr);
    // the ghosts' slopes from the boundary cells'
    if (rowv && (c == -1 || c + 1 == n)) {
        double g[4];
        L.ghost_slope_near(c == -1, c == -1 ? sr : s, g);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (c == -1) s[q] = g[q]; else sr[q] = g[q];
        }
    }

    double F[4] = {0.0, 0.0, 0.0, 0.0}, I[4] = {0.0, 0.0, 0.0, 0.0};
    const int f = c + 1;
    const bool face = rowv && f <= n;
    double pg = -1.0;
    if constexpr (LEARNED) {
        const Side SL = recon(w, s, hh, true);
        const Side SR = recon(wr, sr, hh, false);
        pg = interface_guess<DIR>(src.get(), face, SL, SR, mlp);
    }
    if (face) {
        // the argument block is read again here and after the solve, so that
        // none of it is held across the solve
        const Side SL = recon(w, s, hh, true);
        const Side SR = recon(wr, sr, hh, false);
        solve_interface<DIR, NM, MINW>(src.get(), src, SL, SR, j, f, F, I, tab, pg);
    }
    double Fl[4], Il[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) { Fl[q] = __shfl_up(F[q], STEP); Il[q] = __shfl_up(I[q], STEP); }
    if (k >= 1 && own) {
        const SweepArgs ar = src.get();
        const Line<DIR> Lr(ar, j);
        double wc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) wc[q] = st[q][lane];
        Lr.update(c, wc, st[4][lane], Fl, F, Il, I);
    }
}

// X and Y sweeps (wave_sweep): blocks of 4 waves, wave index = global wave number.
template <int MINW, int NM, int G>
__global__ void __launch_bounds__(256, MINW) sweep_x_kernel(SweepArgs a, int per_row)
{
    constexpr bool LEARNED = NM == NM_LEARNED;
    __shared__ uint32_t mlp_lds[LEARNED ? 4 : 1][LEARNED ? 64 * 8 : 1];
    __shared__ double stash[4][5][64];   // each wave's cell values and E, read back for the update
    __shared__ double tab[POW_TAB];
    const int wv = (threadIdx.x >> 6) & 3;
    const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    wave_sweep<0, MINW, NM, G>(a, KernargArgs{}, wave, per_row, stash[wv], mlp_lds[wv], tab);
}

template <int MINW, int NM, int G>
__global__ void __launch_bounds__(256, MINW) sweep_y_kernel(SweepArgs a, int per_row)
{
    constexpr bool LEARNED = NM == NM_LEARNED;
    __shared__ uint32_t mlp_lds[LEARNED ? 4 : 1][LEARNED ? 64 * 8 : 1];
    __shared__ double stash[4][5][64];
    __shared__ double tab[POW_TAB];
    const int wv = (threadIdx.x >> 6) & 3;
    const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    wave_sweep<1, MINW, NM, G>(a, KernargArgs{}, wave, per_row, stash[wv], mlp_lds[wv], tab);
}

}  // namespace hgrp
