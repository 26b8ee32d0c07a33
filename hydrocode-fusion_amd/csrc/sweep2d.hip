// sweep2d.hip -- gfx950 kernels of the dimension-split 2D GRP step.
//
//   sweep_x_kernel   one X(tau_s) sweep, sweep_y_kernel one Y(tau) sweep: a wave
//                    holds 64/G grid lines of G consecutive cells along the sweep
//                    and exchanges neighbour values, slopes and fluxes with lane
//                    shuffles (wave_sweep).
// Each kernel takes the Newton mode (NM_*) as a template argument.
//   cfl_kernel       h/S_max over the frozen initial data (order-independent min).
//
// Semantics follow src/finite_volume/grp_solver_2D_split_EUL_source.c:182-303,
// src/inter_process/bound_cond_slope_limiter_{x,y}.c:27-129,
// src/inter_process/slope_limiter{,_2D_x}.c and src/flux_calc/flux_generator_{x,y}.c:31-165.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include "grp_device.hpp"
#include "sweep2d.hpp"
#include "sweep2d_body.hpp"

namespace hgrp {

// min over cells of min(h_x, h_y) / (|c| + |u| + |v|)  (grp_solver_2D_split_EUL_source.c:185-191).
// fmin is exact, so the order of the reduction does not matter; positive
// doubles order like their bit patterns, so a 64-bit atomicMin reduces them.
__global__ void __launch_bounds__(256) cfl_kernel(const double *rho, const double *u, const double *v,
                                                  const double *p, int m, int n, int ld, double gamma,
                                                  double hmin, unsigned long long *out)
{
    double best = INFINITY;
    const long total = (long)m * n;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (long)gridDim.x * blockDim.x) {
        const long j = k / n, i = k % n;
        const size_t o = (size_t)j * ld + i;
        const double c = sqrt(gamma * p[o] / rho[o]);
        const double sigma = fabs(c) + fabs(u[o]) + fabs(v[o]);
        best = fmin(best, hmin / sigma);
    }
    for (int off = 32; off > 0; off >>= 1) best = fmin(best, __shfl_xor(best, off));
    if ((threadIdx.x & 63) == 0) {
        unsigned long long bits = __double_as_longlong(best);
        if (!(best >= 0.0)) bits = 0x7ff0000000000000ull;   // NaN never wins a fmin
        atomicMin(out, bits);
    }
}

// ---- launchers -----------------------------------------------------------------
// The launch variants (sweep_shape): the tuner, hgrp2d_tune, times them on the
// context's own data.
int sweep_variants(int dir) { return dir == 0 ? 6 : 5; }
int default_sweep(int dir, int m, int n) { return default_variant(dir, m, n); }

// the variants of three waves per SIMD (sweep2d_few.hip)
hipError_t launch_sweep_few(int dir, const SweepArgs &a, int variant, hipStream_t st);

template <int NM>
static hipError_t launch_x(const SweepArgs &a, int v, hipStream_t st)
{
    const WaveGrid w = wave_grid(0, a.m, a.n, sweep_shape(0, v).G);
    const dim3 grid((unsigned)w.blocks), block(256);
    switch (v) {
    case 1: hipLaunchKernelGGL((sweep_x_kernel<4, NM, 32>), grid, block, 0, st, a, w.per_row); break;
    case 2: hipLaunchKernelGGL((sweep_x_kernel<4, NM, 8>), grid, block, 0, st, a, w.per_row); break;
    case 4: hipLaunchKernelGGL((sweep_x_kernel<4, NM, 4>), grid, block, 0, st, a, w.per_row); break;
    default: hipLaunchKernelGGL((sweep_x_kernel<4, NM, 16>), grid, block, 0, st, a, w.per_row); break;
    }
    return hipGetLastError();
}

template <int NM>
static hipError_t launch_y(const SweepArgs &a, int v, hipStream_t st)
{
    const WaveGrid w = wave_grid(1, a.m, a.n, sweep_shape(1, v).G);
    const dim3 grid((unsigned)w.blocks), block(256);
    switch (v) {
    case 1: hipLaunchKernelGGL((sweep_y_kernel<4, NM, 32>), grid, block, 0, st, a, w.per_row); break;
    case 2: hipLaunchKernelGGL((sweep_y_kernel<4, NM, 64>), grid, block, 0, st, a, w.per_row); break;
    case 3: hipLaunchKernelGGL((sweep_y_kernel<4, NM, 8>), grid, block, 0, st, a, w.per_row); break;
    default: hipLaunchKernelGGL((sweep_y_kernel<4, NM, 16>), grid, block, 0, st, a, w.per_row); break;
    }
    return hipGetLastError();
}

hipError_t launch_sweep_x(const SweepArgs &a, int variant, hipStream_t st)
{
    if (sweep_shape(0, variant).minw == 3) return launch_sweep_few(0, a, variant, st);
    switch (newton_mode(a)) {
    case NM_LEARNED: return launch_x<NM_LEARNED>(a, variant, st);
    case NM_CONV: return launch_x<NM_CONV>(a, variant, st);
    default: return launch_x<NM_REF>(a, variant, st);
    }
}

hipError_t launch_sweep_y(const SweepArgs &a, int variant, hipStream_t st)
{
    if (sweep_shape(1, variant).minw == 3) return launch_sweep_few(1, a, variant, st);
    switch (newton_mode(a)) {
    case NM_LEARNED: return launch_y<NM_LEARNED>(a, variant, st);
    case NM_CONV: return launch_y<NM_CONV>(a, variant, st);
    default: return launch_y<NM_REF>(a, variant, st);
    }
}

// the kernel's name as profilers print it
const char *sweep_kernel_name(int dir, int variant, int nm)
{
#define HGRP_NAMES(k, w, g) {k "<" #w ", 0, " #g ">", k "<" #w ", 1, " #g ">", k "<" #w ", 2, " #g ">"}
    static const char *xn[6][3] = {HGRP_NAMES("sweep_x_kernel", 4, 16), HGRP_NAMES("sweep_x_kernel", 4, 32),
                                   HGRP_NAMES("sweep_x_kernel", 4, 8),  HGRP_NAMES("sweep_x_kernel", 3, 16),
                                   HGRP_NAMES("sweep_x_kernel", 4, 4),  HGRP_NAMES("sweep_x_kernel", 3, 32)};
    static const char *yn[5][3] = {HGRP_NAMES("sweep_y_kernel", 4, 16), HGRP_NAMES("sweep_y_kernel", 4, 32),
                                   HGRP_NAMES("sweep_y_kernel", 4, 64), HGRP_NAMES("sweep_y_kernel", 4, 8),
                                   HGRP_NAMES("sweep_y_kernel", 3, 16)};
#undef HGRP_NAMES
    if (nm < 0 || nm > 2 || variant < 0 || variant >= sweep_variants(dir)) return "";
    return dir == 0 ? xn[variant][nm] : yn[variant][nm];
}

hipError_t launch_cfl(const double *rho, const double *u, const double *v, const double *p, int m, int n,
                      int ld, double gamma, double hmin, unsigned long long *out, hipStream_t st)
{
    const long total = (long)m * n;
    long blocks = (total + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(cfl_kernel, dim3((unsigned)blocks), dim3(256), 0, st, rho, u, v, p, m, n, ld, gamma, hmin, out);
    return hipGetLastError();
}

}  // namespace hgrp
