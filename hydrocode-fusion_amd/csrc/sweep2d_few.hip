// sweep2d_few.hip -- the sweeps' launch variants of three waves per SIMD
// (sweep_shape), for grids that have no more to give.  A file of its own because
// it is compiled otherwise than sweep2d.hip (see the Makefile).
#include <hip/hip_runtime.h>
#include "grp_device.hpp"
#include "sweep2d.hpp"
#include "sweep2d_body.hpp"

namespace hgrp {

template <int NM>
static hipError_t launch_few(int dir, const SweepArgs &a, int v, hipStream_t st)
{
    const WaveGrid w = wave_grid(dir, a.m, a.n, sweep_shape(dir, v).G);
    const dim3 grid((unsigned)w.blocks), block(256);
    if (dir == 1) hipLaunchKernelGGL((sweep_y_kernel<3, NM, 16>), grid, block, 0, st, a, w.per_row);
    else if (v == 3) hipLaunchKernelGGL((sweep_x_kernel<3, NM, 16>), grid, block, 0, st, a, w.per_row);
    else hipLaunchKernelGGL((sweep_x_kernel<3, NM, 32>), grid, block, 0, st, a, w.per_row);
    return hipGetLastError();
}

hipError_t launch_sweep_few(int dir, const SweepArgs &a, int variant, hipStream_t st)
{
    switch (newton_mode(a)) {
    case NM_LEARNED: return launch_few<NM_LEARNED>(dir, a, variant, st);
    case NM_CONV: return launch_few<NM_CONV>(dir, a, variant, st);
    default: return launch_few<NM_REF>(dir, a, variant, st);
    }
}

}  // namespace hgrp
