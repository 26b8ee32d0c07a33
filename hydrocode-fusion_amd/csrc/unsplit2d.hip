// unsplit2d.hip -- the genuinely 2D GRP step (no dimension splitting), one
// launch per time step.
//
//   unsplit_step_kernel  a wave covers a tile of 7 x 8 cells.  It forms the "side
//                        data" of the tile's cells and of those around it --
//                        value, limited x-slope, limited y-slope, or the ghost's
//                        value and slopes at the edges -- in its LDS slots, solves
//                        the tile's y-interfaces, then its x-interfaces, one lane
//                        an interface, and updates the cells with both flux
//                        differences.  Interfaces on tile edges are solved by both
//                        tiles, everything else once.
//
// Semantics follow src/finite_volume/grp_solver_2D_EUL_source.c:181-262,
// src/inter_process/bound_cond_slope_limiter_{x,y}.c:27-129 (including the
// ghost slopes across directions, :111-126) and
// src/flux_calc/flux_generator_{x,y}.c:31-165 with Transversal = true.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include "grp_device.hpp"
#include "g2d_device.hpp"
#include "unsplit2d.hpp"

namespace hgrp {

namespace {

// Values, limited slopes and interface side data around one step.  Rows c
// (x index) run over [-1, m], columns ci (y index) over [-1, n]; -1, m and n
// are ghost cells.
struct Grid {
    const UnsplitArgs &a;
    __device__ explicit Grid(const UnsplitArgs &args) : a(args) {}

    __device__ __forceinline__ size_t at(int c, int ci) const { return (size_t)c * (size_t)a.ld + (size_t)ci; }
    __device__ __forceinline__ void cell(int c, int ci, double w[4]) const
    {
        const size_t o = at(c, ci);
        const double *f = a.st + o;
        w[0] = f[0]; w[1] = f[a.plane]; w[2] = f[2 * a.plane]; w[3] = f[3 * a.plane];
    }
    // value of row c in [-1, m] of column ci in [0, n): x-ghosts per config[17]
    // (bound_cond_slope_limiter_x.c:34-82)
    __device__ __forceinline__ void xval(int c, int ci, double w[4]) const
    {
        if (c >= 0 && c < a.m) { cell(c, ci, w); return; }
        const bool lo = c < 0;
        switch (a.bc_x) {
        case BC_INITIAL: {
            const double *b = (lo ? a.bx_lo : a.bx_hi) + (size_t)ci * 4;
            w[0] = b[0]; w[1] = b[1]; w[2] = b[2]; w[3] = b[3];
            return;
        }
        case BC_PERIODIC: cell(lo ? a.m - 1 : 0, ci, w); return;
        case BC_REFLECT: cell(lo ? 0 : a.m - 1, ci, w); w[1] = -w[1]; return;
        case BC_REFLECT_FREE: cell(lo ? 0 : a.m - 1, ci, w); if (lo) w[1] = -w[1]; return;
        default: cell(lo ? 0 : a.m - 1, ci, w); return;
        }
    }
    // value of column ci in [-1, n] of row c in [0, m): y-ghosts per config[18]
    // (bound_cond_slope_limiter_y.c:34-82)
    __device__ __forceinline__ void yval(int c, int ci, double w[4]) const
    {
        if (ci >= 0 && ci < a.n) { cell(c, ci, w); return; }
        const bool lo = ci < 0;
        switch (a.bc_y) {
        case BC_INITIAL: {
            const double *b = (lo ? a.by_lo : a.by_hi) + (size_t)c * 4;
            w[0] = b[0]; w[1] = b[1]; w[2] = b[2]; w[3] = b[3];
            return;
        }
        case BC_PERIODIC: cell(c, lo ? a.n - 1 : 0, w); return;
        case BC_REFLECT: cell(c, lo ? 0 : a.n - 1, w); w[2] = -w[2]; return;
        case BC_REFLECT_FREE: cell(c, lo ? 0 : a.n - 1, w); if (lo) w[2] = -w[2]; return;
        default: cell(c, lo ? 0 : a.n - 1, w); return;
        }
    }
    // minmod slope from the neighbours (slope_limiter_2D_x.c:32-84, slope_limiter.c:31-83)
    __device__ __forceinline__ void limit(const double vm[4], const double v0[4], const double vp[4], const double *prev,
                          size_t o, int lim3, const RecipDiv &d, double s[4]) const
    {
        double d_L[4], d_R[4], s_L[4], s_R[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) { d_L[q] = v0[q] - vm[q]; d_R[q] = vp[q] - v0[q]; }
        quot4(d_L, d, s_L);
        quot4(d_R, d, s_R);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            s[q] = lim3 ? minmod3(a.alpha * s_L[q], a.alpha * s_R[q], prev[o + q * a.plane]) : minmod2(s_L[q], s_R[q]);
    }

    // Side data of (c, ci): value v, x-slope s, y-slope t.  A cell: its limited
    // slopes.  An x-ghost (c = -1 or m): bfv_L/R -- ghost value, the x-slope
    // rule of bound_cond_slope_limiter_x.c:94-109 and, across, the y-slopes of
    // the boundary cell (bound_cond_slope_limiter_y.c:111-126).  A y-ghost
    // (ci = -1 or n): bfv_D/U with the mirrored rules.  Slopes the reference
    // never sets stay zero (its ghost arrays are calloc'ed).  Not for corners.
    // Every ghost takes what it takes from one cell: the one next to it, or the
    // last one of the line with periodic ends; so one limiter serves all.
    __device__ __forceinline__ void side(int c, int ci, double v[4], double s[4], double t[4]) const
    {
        const bool xin = c >= 0 && c < a.m, yin = ci >= 0 && ci < a.n;
        const bool lo = c < 0 || ci < 0;
        const int bc = xin ? a.bc_y : a.bc_x;                 // of a ghost
        const bool far = bc == BC_PERIODIC;
        const int cs = xin ? c : (lo != far ? 0 : a.m - 1), is = yin ? ci : (lo != far ? 0 : a.n - 1);
        double v0[4], vm[4], vp[4];
        cell(cs, is, v0);
        xval(cs - 1, is, vm);
        xval(cs + 1, is, vp);
        limit(vm, v0, vp, a.s, at(cs, is), a.lim3_x, a.div_hx, s);
        yval(cs, is - 1, vm);
        yval(cs, is + 1, vp);
        limit(vm, v0, vp, a.t, at(cs, is), a.lim3_y, a.div_hy, t);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = v0[q];
        if (!(xin && yin)) {
            // the normal velocity and its slope across the boundary that the ghost lies behind
            const bool mirror = bc == BC_REFLECT || (bc == BC_REFLECT_FREE && lo);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool normal = q == (xin ? 2 : 1);
                if (mirror && normal) v[q] = -v[q];
                if (!(far || (mirror && normal))) { if (xin) t[q] = 0.0; else s[q] = 0.0; }
                if (bc == BC_INITIAL) { if (xin) s[q] = 0.0; else t[q] = 0.0; }
            }
            if (bc == BC_INITIAL) {
                if (xin) yval(c, ci, v); else xval(c, ci, v);
            }
        }
    }
};

// GRP solve of one interface with transversal derivatives, normal x (dir 0)
// or y (dir 1); failures are recorded in status[dir] as
// ((loop index << 2) | code) + 1, the reference's loop order
// G2: GRP_2D_flux with its alternative solver, G2D (grp_2d_flux_g2d).
// (c, ci): the cell on its left (lower) side.

// The face with the IEEE solver, from the cells in memory: what the fast solver
// leaves (grp_fast.hpp).
template <int NM>
__device__ __attribute__((noinline)) int redo_face_t(const UnsplitArgs *ap, int dir, int c, int ci, double p_guess,
                                                     double *FI)
{
    const UnsplitArgs &a = *ap;
    const Grid G(a);
    double vl[4], sl[4], tl[4], vr[4], sr[4], tr[4];
    G.side(c, ci, vl, sl, tl);
    G.side(dir ? c : c + 1, dir ? ci + 1 : ci, vr, sr, tr);
    if (dir) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            double x = sl[q];
            sl[q] = tl[q]; tl[q] = -x;
            x = sr[q];
            sr[q] = tr[q]; tr[q] = -x;
        }
    }
    const double hh = dir ? a.hh_y : a.hh_x;
    return grp_2d_flux_n<NM != NM_REF>(recon(vl, sl, hh, true), recon(vr, sr, hh, false), tl, tr, a.gas, dir ? 0.0 : 1.0,
                                       dir ? 1.0 : 0.0, a.tau, a.eps, FI, FI + 4, a.tol, p_guess);
}

template <int NM, bool G2>
__device__ __forceinline__ void solve_t(const UnsplitArgs &a, int dir, const Side &SL, const Side &SR,
                                        const double TL[4], const double TR[4], int c, int ci, double F[4], double I[4],
                                        double p_guess, const double *tab)
{
    int code = ifvar_bad_t(SL, SR, TL, TR, a.eps) ? 1 : 0, bad = 0;
    const double n_x = dir ? 0.0 : 1.0, n_y = dir ? 1.0 : 0.0;
    if constexpr (G2) {
        bad = grp_2d_flux_g2d<NM != NM_REF>(SL, SR, TL, TR, a.gas, n_x, n_y, a.tau, a.eps, F, I, a.tol, p_guess, tab);
    } else {
        const bool done = flux_transversal_q<NM != NM_REF>(SL, SR, TL, TR, a.gas, dir, a.near2, a.tau, a.eps, F, I, a.tol,
                                                           p_guess, &bad, tab);
        if (__builtin_expect(__any(!done), 0)) {
            if (!done) {
                const UnsplitArgs ar = reload_args<UnsplitArgs>();
                double o[8];
                bad = redo_face_t<NM>(&ar, dir, c, ci, p_guess, o);
#pragma unroll
                for (int q = 0; q < 4; ++q) { F[q] = o[q]; I[q] = o[4 + q]; }
            }
        }
    }
    if (bad) code = 2;
    if (code) {
        const UnsplitArgs ar = reload_args<UnsplitArgs>();
        const unsigned long long index =
            dir ? (unsigned long long)c * (unsigned long long)(ar.n + 1) + (unsigned long long)(ci + 1)
                : (unsigned long long)ci * (unsigned long long)(ar.m + 1) + (unsigned long long)(c + 1);
        atomicMax(&ar.status[dir].fail_key, ((index << 2) | (unsigned long long)code) + 1ull);
    }
}

// Learned starting pressure for the interface (SL | SR) with normal x (dir 0)
// or y (dir 1), every lane of the wave (uniform call); -1 outside NM_LEARNED,
// where Newton will not run (the acoustic shortcut, the equal-state exit) or
// where the lane has no interface.  The states are those normal to the
// interface (GRP_2D_flux's rotation keeps rho and p; u_n is u or v).
template <int NM>
__device__ __forceinline__ double unsplit_guess(const UnsplitArgs &a, bool active, int dir, const Side &SL,
                                                const Side &SR, uint32_t *lds)
{
    if constexpr (NM != NM_LEARNED) {
        return -1.0;
    } else {
        const double uL = dir ? SL.v : SL.u, uR = dir ? SR.v : SR.u;
        const double dist2 = (SL.rho - SR.rho) * (SL.rho - SR.rho) + (uL - uR) * (uL - uR)
                             + (SL.p - SR.p) * (SL.p - SR.p);
        const bool want = active && !(dist2 < a.near2) && !(fabs(uL - uR) < a.tol && fabs(SL.p - SR.p) < a.tol);
        return learned_guess_wave(a.mlp, want, SL.rho, uL, SL.p, SR.rho, uR, SR.p, a.gas.g, a.gas.g, lds);
    }
}

}  // namespace

// Tile form: a wave owns a tile of 7 x 8 cells (rows along x, columns along y).
// Its 8 x 8 x-interfaces fill the wave, its 7 x 9 y-interfaces all but a lane;
// the side data of its 9 x 10 cells lie in the wave's own LDS slots, and the
// faces go to the cells' lanes by shuffles, so no wave waits for another once
// the pow tables are there.  (A tile of 12 waves, 10 rows of 62 cells, handed its
// faces on through 160 KiB of LDS, one block to a CU, and waited 58 % of its time
// at the barriers.  A step with it and with this: 300^2 .062 and .054 ms, 512^2
// .108 and .092, 1024^2 .281 and .283, 4096^2 3.84 and 3.22; G2D 257 x 190 .089
// and .049, 1024^2 .337 and .347.)
// Of 8 or 9 cells in x the second row of such tiles holds one or two; a tile of 9
// x 6 (10 x 6 and 9 x 7 interfaces) takes them all (tile_shape).
template <int SHAPE>
struct Tile {
    static constexpr int R = SHAPE == 1 ? 7 : 9, C = SHAPE == 1 ? 8 : 6;
    static constexpr int SIDE_C = C + 2, SIDES = (R + 2) * SIDE_C - 1;   // not the last corner
    static constexpr int XF = (R + 1) * C, YF = R * (C + 1);             // interfaces, a lane each
    static_assert(XF <= 64 && YF <= 64, "a lane to an interface");
};

template <int SHAPE, int NM, bool G2>
__device__ __forceinline__ void unsplit_step_body(const UnsplitArgs &a, int per_row)
{
    constexpr bool LEARNED = NM == NM_LEARNED;
    constexpr int R = Tile<SHAPE>::R, C = Tile<SHAPE>::C, SIDE_C = Tile<SHAPE>::SIDE_C, SIDES = Tile<SHAPE>::SIDES;
    constexpr int XF = Tile<SHAPE>::XF, YF = Tile<SHAPE>::YF;
    __shared__ double sides_lds[4][12][SIDES];   // value, x-slope, y-slope of the tile's cells and the ones around
    __shared__ double tab[POW_TAB];
    __shared__ uint32_t mlp_lds[LEARNED ? 4 : 1][LEARNED ? 64 * 8 : 1];
    const int lane = threadIdx.x & 63, wv = (threadIdx.x >> 6) & 3;
    const long wave = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int j0 = (int)(wave / per_row) * R, i0 = (int)(wave % per_row) * C;
    double(*sd)[SIDES] = sides_lds[wv];
    // the lane's cell (row r, column k of the tile with its halo; updated for r >= 1) and x-interface,
    // between rows r and r + 1
    const int r = lane / C, k = lane % C + 1, c = j0 - 1 + r, ci = i0 - 1 + k;
    const bool own = r >= 1 && lane < XF && c < a.m && ci < a.n;
    {
        const Grid G(a);
        TabLoad<256> tl;
        tl.load(threadIdx.x);
#pragma unroll 1
        for (int id = lane; id < SIDES; id += 64) {
            const int sc = j0 - 1 + id / SIDE_C, si = i0 - 1 + id % SIDE_C;
            double v[4] = {1.0, 0.0, 0.0, 1.0}, s[4] = {0.0, 0.0, 0.0, 0.0}, t[4] = {0.0, 0.0, 0.0, 0.0};
            const bool xin = sc >= 0 && sc < a.m, yin = si >= 0 && si < a.n;
            if (sc <= a.m && si <= a.n && (xin || yin)) G.side(sc, si, v, s, t);   // a cell or a ghost, not a corner
#pragma unroll
            for (int q = 0; q < 4; ++q) { sd[q][id] = v[q]; sd[4 + q][id] = s[q]; sd[8 + q][id] = t[q]; }
        }
        // a failed step ends the run: later steps do nothing.  The status is read
        // after the side loads went out (they stay in bounds either way); the
        // whole block returns together.
        if (a.prev != nullptr) {
            const SweepStatus p0 = a.prev[0], p1 = a.prev[1];
            if (p0.fail_key != 0ull || p0.flags != 0u || p1.fail_key != 0ull) {
                if (threadIdx.x == 0) atomicOr(&a.status[0].flags, 2u);
                return;
            }
        }
        tl.store(threadIdx.x, tab);
    }
    __syncthreads();
    if (j0 >= a.m) return;                                   // a wave past the last tile

    // dir 1: y-interfaces of the updated rows (flux_generator_y.c:42-121), normal derivative =
    //        y-slope, transversal = -(x-slope);
    // dir 0: x-interface f = c + 1 between rows c and c + 1 (flux_generator_x.c:42-121).
    // One solve site for both, so the GRP code and its registers are laid out once.
    const int yr = lane / (C + 1) + 1, yk = lane % (C + 1), yc = j0 - 1 + yr, ycell = i0 - 1 + yk;
    double dG[4];
#pragma unroll 1
    for (int dir = 1; dir >= 0; --dir) {
        const bool active = dir ? lane < YF && yc < a.m && ycell < a.n : lane < XF && c < a.m && ci < a.n;
        const int id0 = dir ? yr * SIDE_C + yk : r * SIDE_C + k, id1 = dir ? id0 + 1 : id0 + SIDE_C;
        Side SL, SR;
        double TL[4], TR[4];
        // the two cells' side data: value, normal and transversal slope
        auto sides = [&]() {
            const int sn = dir ? 8 : 4, st = dir ? 4 : 8;
            const double hh = dir ? a.hh_y : a.hh_x;
            double vl[4], sl[4], vr[4], sr[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                vl[q] = sd[q][id0]; sl[q] = sd[sn + q][id0]; TL[q] = sd[st + q][id0];
                vr[q] = sd[q][id1]; sr[q] = sd[sn + q][id1]; TR[q] = sd[st + q][id1];
            }
            if (dir)
#pragma unroll
                for (int q = 0; q < 4; ++q) { TL[q] = -TL[q]; TR[q] = -TR[q]; }
            SL = recon(vl, sl, hh, true);
            SR = recon(vr, sr, hh, false);
        };
        double F[4] = {0.0, 0.0, 0.0, 0.0}, I[4] = {0.0, 0.0, 0.0, 0.0}, pg = -1.0;
        if constexpr (LEARNED) {   // a call: the sides are read again after it, not held across
            if (active) sides();
            pg = unsplit_guess<NM>(a, active, dir, SL, SR, mlp_lds[wv]);
        }
        // the argument block is read again for the solve, so no scalar register holds it across
        if (active) {
            sides();
            solve_t<NM, G2>(reload_args<UnsplitArgs>(), dir, SL, SR, TL, TR, dir ? yc : c, dir ? ycell : ci, F, I, pg, tab);
        }
        const UnsplitArgs a = reload_args<UnsplitArgs>();
        const size_t o = (size_t)c * (size_t)a.ld + (size_t)ci, P = a.plane;
        if (dir) {   // the y-faces on both sides of the lane's cell
            const int hi = r >= 1 && lane < XF ? (r - 1) * (C + 1) + k : 1;
            double dI[4], tn[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                dG[q] = __shfl(F[q], hi) - __shfl(F[q], hi - 1);
                dI[q] = __shfl(I[q], hi) - __shfl(I[q], hi - 1);
            }
            if (own) {
                quot4(dI, a.div_hy, tn);
#pragma unroll
                for (int q = 0; q < 4; ++q) a.t_o[o + q * P] = tn[q];
            }
            continue;
        }
        // combined update and slope refresh (grp_solver_2D_EUL_source.c:231-262)
        double dF[4], dI[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            dF[q] = F[q] - __shfl_up(F[q], C);
            dI[q] = I[q] - __shfl_up(I[q], C);
        }
        if (own) {
            const double e_c = a.st[o + 4 * P];
            double vc[4], sn[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) vc[q] = sd[q][id0];
            const double nu = a.nu, mu = a.mu;
            const double mom_x = vc[0] * vc[1] - nu * dF[1] - mu * dG[1];
            const double mom_y = vc[0] * vc[2] - nu * dF[2] - mu * dG[2];
            const double ene = vc[0] * e_c - nu * dF[3] - mu * dG[3];
            const double rho = vc[0] + (-nu * dF[0] - mu * dG[0]);
            double uu, vv, e_new;
            quot3(mom_x, mom_y, ene, rho, uu, vv, e_new);
            const double p = (ene - 0.5 * mom_x * uu - 0.5 * mom_y * vv) * a.gas.gm1();
            double *fo = a.st_o + o;
            fo[0] = rho; fo[P] = uu; fo[2 * P] = vv; fo[4 * P] = e_new; fo[3 * P] = p;
            if (p < a.eps || rho < a.eps) atomicOr(&a.status[0].flags, 1u);
            quot4(dI, a.div_hx, sn);
#pragma unroll
            for (int q = 0; q < 4; ++q) a.s_o[o + q * P] = sn[q];
        }
    }
}

// CU_WAVES: the waves that the register budget lets a CU hold; SHAPE: the tile's
// (1: 7 x 8, 2: 9 x 6).
template <int CU_WAVES, int SHAPE, int NM>
__global__ void __launch_bounds__(256, CU_WAVES / 4) unsplit_step_kernel(UnsplitArgs a, int per_row)
{
    unsplit_step_body<SHAPE, NM, false>(a, per_row);
}

// the same step with GRP_2D_flux's alternative interface solver, G2D
template <int CU_WAVES, int SHAPE, int NM>
__global__ void __launch_bounds__(256, CU_WAVES / 4) unsplit_step_g2d_kernel(UnsplitArgs a, int per_row)
{
    unsplit_step_body<SHAPE, NM, true>(a, per_row);
}

// Strip form: one wave per block walks down R cell rows of a 62-cell strip
// (lanes: cells i0-1 .. i0+62 of the row).  Iteration r (from r0-1) forms the
// side data of row r+1, solves the y-interfaces of row r and the x-interface
// r+1 (one solve site, two passes), and updates row r from the x-interface r
// kept from the iteration before.  No wave waits for another: the block is
// one wave, its LDS holds two rows of side data and two rows of interface
// results (16 KiB).  One extra x-interface per R rows.
template <int NM, bool G2>
__device__ __forceinline__ void unsplit_strip_body(const UnsplitArgs &a, int R)
{
    __shared__ double sd[2][12][64];   // side data of rows r and r + 1 (alternating)
    __shared__ double fl[8][64];       // x-interface r: flux, values at t + tau
    __shared__ double gb[8][64];       // y-interfaces of row r: flux, values at t + tau
    __shared__ uint32_t mlp_lds[NM == NM_LEARNED ? 64 * 8 : 1];   // network inputs
    __shared__ double tab[POW_TAB];
    if (a.prev != nullptr) {
        const SweepStatus p0 = a.prev[0], p1 = a.prev[1];
        if (p0.fail_key != 0ull || p0.flags != 0u || p1.fail_key != 0ull) {
            if (threadIdx.x == 0) atomicOr(&a.status[0].flags, 2u);
            return;
        }
    }
    const int lane = threadIdx.x;
    const int m = a.m, n = a.n;
    const int ci = blockIdx.x * 62 - 1 + lane;
    const int r0 = blockIdx.y * R, r1 = min(r0 + R, m);   // rows r0 .. r1-1 are updated here
    const Grid G(a);
    const bool yin = ci >= 0 && ci < n;
    const bool colv = ci <= n;                             // a cell or a y-ghost column

    auto put_side = [&](int buf, int c) {
        double v[4] = {1.0, 0.0, 0.0, 1.0}, s[4] = {0.0, 0.0, 0.0, 0.0}, t[4] = {0.0, 0.0, 0.0, 0.0};
        const UnsplitArgs ar = reload_args<UnsplitArgs>();   // nothing of the loads is held across the solves
        if (colv && c <= m && ((c >= 0 && c < m) || yin)) Grid(ar).side(c, ci, v, s, t);
#pragma unroll
        for (int q = 0; q < 4; ++q) { sd[buf][q][lane] = v[q]; sd[buf][4 + q][lane] = s[q]; sd[buf][8 + q][lane] = t[q]; }
    };
    TabLoad<64> tl;
    tl.load(lane);
    tl.store(lane, tab);
    int cb = 0;
    put_side(cb, r0 - 1);
#pragma unroll 1
    for (int r = r0 - 1; r < r1; ++r) {
        const int nb = 1 - cb;
        put_side(nb, r + 1);
        __syncthreads();
        const bool xin = r >= r0;                          // row r is updated (r0 <= r < r1 <= m)
        double F[4], I[4];
#pragma unroll 1
        for (int pass = 0; pass < 2; ++pass) {
            Side SL, SR;
            double TL[4], TR[4];
            bool active;
            if (pass == 0) {   // y-interface ci + 1 of row r: normal = y-slope, transversal = -(x-slope)
                active = xin && lane <= 62 && ci <= n - 1;
                if (active) {
                    double vd[4], td[4], vu[4], tu[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        vd[q] = sd[cb][q][lane];     td[q] = sd[cb][8 + q][lane];     TL[q] = -sd[cb][4 + q][lane];
                        vu[q] = sd[cb][q][lane + 1]; tu[q] = sd[cb][8 + q][lane + 1]; TR[q] = -sd[cb][4 + q][lane + 1];
                    }
                    SL = recon(vd, td, a.hh_y, true);
                    SR = recon(vu, tu, a.hh_y, false);
                }
            } else {           // x-interface r + 1 between rows r and r + 1
                active = lane >= 1 && lane <= 62 && yin && r + 1 <= m;
                if (active) {
                    double vl[4], sl[4], vr[4], sr[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        vl[q] = sd[cb][q][lane]; sl[q] = sd[cb][4 + q][lane]; TL[q] = sd[cb][8 + q][lane];
                        vr[q] = sd[nb][q][lane]; sr[q] = sd[nb][4 + q][lane]; TR[q] = sd[nb][8 + q][lane];
                    }
                    SL = recon(vl, sl, a.hh_x, true);
                    SR = recon(vr, sr, a.hh_x, false);
                }
            }
            double Fo[4] = {0.0, 0.0, 0.0, 0.0}, Io[4] = {0.0, 0.0, 0.0, 0.0};
            const double pg = unsplit_guess<NM>(a, active, 1 - pass, SL, SR, mlp_lds);
            if (active) solve_t<NM, G2>(reload_args<UnsplitArgs>(), 1 - pass, SL, SR, TL, TR, r, ci, Fo, Io, pg, tab);
            if (pass == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) { gb[q][lane] = Fo[q]; gb[4 + q][lane] = Io[q]; }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) { F[q] = Fo[q]; I[q] = Io[q]; }
        }
        __syncthreads();
        if (xin && yin && lane >= 1 && lane <= 62) {
            const UnsplitArgs a = reload_args<UnsplitArgs>();
            const size_t o = G.at(r, ci);
            const double e_c = a.st[o + 4 * a.plane];
            double vc[4], Fl[4], Ixl[4], Gy[4], Gl[4], Iy[4], Iyl[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                vc[q] = sd[cb][q][lane];
                Fl[q] = fl[q][lane]; Ixl[q] = fl[4 + q][lane];
                Gy[q] = gb[q][lane]; Iy[q] = gb[4 + q][lane];
                Gl[q] = gb[q][lane - 1]; Iyl[q] = gb[4 + q][lane - 1];
            }
            const double nu = a.nu, mu = a.mu;
            const double mom_x = vc[0] * vc[1] - nu * (F[1] - Fl[1]) - mu * (Gy[1] - Gl[1]);
            const double mom_y = vc[0] * vc[2] - nu * (F[2] - Fl[2]) - mu * (Gy[2] - Gl[2]);
            const double ene = vc[0] * e_c - nu * (F[3] - Fl[3]) - mu * (Gy[3] - Gl[3]);
            const double rho = vc[0] + (-nu * (F[0] - Fl[0]) - mu * (Gy[0] - Gl[0]));
            double uu, vv, e_new, dx[4], dy[4], sn[4], tn[4];
            quot3(mom_x, mom_y, ene, rho, uu, vv, e_new);
            const double p = (ene - 0.5 * mom_x * uu - 0.5 * mom_y * vv) * a.gas.gm1();
            double *fo = a.st_o + o;
            const size_t P = a.plane;
            fo[0] = rho; fo[P] = uu; fo[2 * P] = vv; fo[4 * P] = e_new; fo[3 * P] = p;
            if (p < a.eps || rho < a.eps) atomicOr(&a.status[0].flags, 1u);
#pragma unroll
            for (int q = 0; q < 4; ++q) { dx[q] = I[q] - Ixl[q]; dy[q] = Iy[q] - Iyl[q]; }
            quot4(dx, a.div_hx, sn);
            quot4(dy, a.div_hy, tn);
#pragma unroll
            for (int q = 0; q < 4; ++q) { a.s_o[o + q * P] = sn[q]; a.t_o[o + q * P] = tn[q]; }
        }
        // x-interface r + 1 is the next row's lower interface (each lane keeps its own slot)
#pragma unroll
        for (int q = 0; q < 4; ++q) { fl[q][lane] = F[q]; fl[4 + q][lane] = I[q]; }
        cb = nb;
    }
}

template <int NM>
__global__ void __launch_bounds__(64, 2) unsplit_strip_kernel(UnsplitArgs a, int R)
{
    unsplit_strip_body<NM, false>(a, R);
}

// the same with GRP_2D_flux's alternative interface solver, G2D
template <int NM>
__global__ void __launch_bounds__(64, 2) unsplit_strip_g2d_kernel(UnsplitArgs a, int R)
{
    unsplit_strip_body<NM, true>(a, R);
}

// ---- launchers -----------------------------------------------------------------
// Two forms: the tile (a wave to a tile of cells) and the strip (one wave per
// block walking down its rows).  The context picks one
// (hgrp2d_set_unsplit_form, hgrp2d_tune) or takes the default (form 0: the tile).
// The tile's register budget is three waves per SIMD (168 VGPRs, 4-83 spilled;
// 38 KiB of LDS for the 4 waves of a block): with two waves and no spills a step
// of 1024^2 takes .333 instead of .283 ms, with four .360.

// rows per strip of the strip form: enough strips to give every CU several waves
static int strip_rows(int m, int n)
{
    const long strips = (long)((n + 61) / 62);
    int R = 32;
    while (R > 4 && strips * ((m + R - 1) / R) < 4L * 2048) R /= 2;
    return R;
}

// Form 0 and 1: the tile, which is the faster at every size measured; 2: the strip.
static bool use_strip(int form) { return form == 2; }

int unsplit_max_rows() { return 65535 * 4; }   // grid.y of the strip form at R = 4

template <int SHAPE>
static long tiles_of(int m, int n)
{
    return (long)((m + Tile<SHAPE>::R - 1) / Tile<SHAPE>::R) * ((n + Tile<SHAPE>::C - 1) / Tile<SHAPE>::C);
}

// The tile's shape: 9 x 6 where the grid has more tiles of 7 x 8 than the chip
// holds waves at once (12 to a CU) and a quarter fewer of 9 x 6, which is so on 8
// and 9 cells in x.  A step of 8 x 31000 with 7 x 8 and with 9 x 6: .144 and .123
// ms, 9 x 16384 .084 and .070; G2D 8 x 31000 .183 and .156.
static int tile_shape(int m, int n)
{
    const long t = tiles_of<1>(m, n);
    return t > 12 * 256 && 4 * tiles_of<2>(m, n) <= 3 * t ? 2 : 1;
}

template <int SHAPE, int NM, bool G2>
static void launch_tile(const UnsplitArgs &a, hipStream_t st)
{
    const int per_row = (a.n + Tile<SHAPE>::C - 1) / Tile<SHAPE>::C;
    const dim3 grid((unsigned)((tiles_of<SHAPE>(a.m, a.n) + 3) / 4));
    if (G2) hipLaunchKernelGGL((unsplit_step_g2d_kernel<12, SHAPE, NM>), grid, dim3(256), 0, st, a, per_row);
    else hipLaunchKernelGGL((unsplit_step_kernel<12, SHAPE, NM>), grid, dim3(256), 0, st, a, per_row);
}

template <int NM, bool G2>
static hipError_t launch_unsplit(const UnsplitArgs &a, hipStream_t st)
{
    if (use_strip(a.form)) {
        const int R = strip_rows(a.m, a.n);
        const dim3 grid((unsigned)((a.n + 61) / 62), (unsigned)((a.m + R - 1) / R));
        if (G2) hipLaunchKernelGGL(unsplit_strip_g2d_kernel<NM>, grid, dim3(64), 0, st, a, R);
        else hipLaunchKernelGGL(unsplit_strip_kernel<NM>, grid, dim3(64), 0, st, a, R);
    } else if (tile_shape(a.m, a.n) == 2) {
        launch_tile<2, NM, G2>(a, st);
    } else {
        launch_tile<1, NM, G2>(a, st);
    }
    return hipGetLastError();
}

template <bool G2>
static hipError_t launch_unsplit_nm(const UnsplitArgs &a, hipStream_t st)
{
    if (a.mlp) return launch_unsplit<NM_LEARNED, G2>(a, st);
    return a.conv ? launch_unsplit<NM_CONV, G2>(a, st) : launch_unsplit<NM_REF, G2>(a, st);
}

hipError_t launch_unsplit_step(const UnsplitArgs &a, hipStream_t st)
{
    return a.g2d ? launch_unsplit_nm<true>(a, st) : launch_unsplit_nm<false>(a, st);
}

const char *unsplit_kernel_name(int m, int n, int nm, int g2d, int form)
{
    static const char *names[2][3][3] = {
        {{"unsplit_step_kernel<12, 1, 0>", "unsplit_step_kernel<12, 2, 0>", "unsplit_strip_kernel<0>"},
         {"unsplit_step_kernel<12, 1, 1>", "unsplit_step_kernel<12, 2, 1>", "unsplit_strip_kernel<1>"},
         {"unsplit_step_kernel<12, 1, 2>", "unsplit_step_kernel<12, 2, 2>", "unsplit_strip_kernel<2>"}},
        {{"unsplit_step_g2d_kernel<12, 1, 0>", "unsplit_step_g2d_kernel<12, 2, 0>", "unsplit_strip_g2d_kernel<0>"},
         {"unsplit_step_g2d_kernel<12, 1, 1>", "unsplit_step_g2d_kernel<12, 2, 1>", "unsplit_strip_g2d_kernel<1>"},
         {"unsplit_step_g2d_kernel<12, 1, 2>", "unsplit_step_g2d_kernel<12, 2, 2>", "unsplit_strip_g2d_kernel<2>"}}};
    if (nm < 0 || nm > 2) return "";
    return names[g2d ? 1 : 0][nm][use_strip(form) ? 2 : tile_shape(m, n) - 1];
}

}  // namespace hgrp
