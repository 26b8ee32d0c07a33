// layout2d.hpp -- copies between a caller's packed m x n arrays and the
// solver's pitched field planes (layout2d.hip).  stage: planes of the same size
// that hold nothing of use (the buffer set that the next sweep overwrites).
// All are enqueued on st.
#pragma once
#include <hip/hip_runtime.h>

namespace hgrp {

// rho u v p (and E, or nullptr: formed on the device) to dst, and the BC -1
// ghost tables from them to bnd (2 n x 4 and 2 m x 4 doubles)
hipError_t upload_state(const double *const src[5], double *stage, double *dst, double *bnd, size_t plane, int m, int n,
                        int ld, double gamma, hipStream_t st);
hipError_t upload_plane(const double *src, double *stage, double *dst, int m, int n, int ld, hipStream_t st);
// nf planes from src, each to dst[f] unless that is nullptr
hipError_t download_planes(double *const dst[], int nf, const double *src, double *stage, size_t plane, int m, int n, int ld,
                           hipStream_t st);

}  // namespace hgrp
