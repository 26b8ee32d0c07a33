// layout2d.hip -- between the caller's packed arrays and the solver's planes.
//
// A host array is m*n doubles, cell (j, i) at j*n + i; a field plane has the
// row pitch ld >= n (sweep2d.hpp).  A strided copy between the two goes row by
// row through the runtime (about 1 GB/s from pageable memory at 1024^2 and
// less on smaller rows), a contiguous one at the link's rate (29 GB/s up, 18
// down).  So the arrays cross as they are, into or out of the buffer set that
// the next sweep overwrites, and these kernels move them to or from their
// pitch on the device; the upload also forms E and the BC -1 ghost tables
// there.  All are bound by HBM and negligible beside the link.  1024^2: upload
// 49 -> 1.5 ms, download 37 -> 4.8 ms.
#include <hip/hip_runtime.h>

#include "layout2d.hpp"

namespace hgrp {

// packed planes (nf fields, `plane` doubles apart) to pitched ones; with
// form_e the fifth is E = 0.5 u^2 + p/(gamma-1)/rho + 0.5 v^2, as the
// reference's main program forms it (src/hydrocode_2D/hydrocode.c:251-252)
__global__ void __launch_bounds__(256) unpack_kernel(const double *src, double *dst, size_t plane, int m, int n, int ld,
                                                     int nf, int form_e, double gamma)
{
    const size_t total = (size_t)m * n;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (size_t)gridDim.x * blockDim.x) {
        const size_t j = k / n, o = j * ld + (k - j * n);
        if (form_e) {
            const double rho = src[k], u = src[plane + k], v = src[2 * plane + k], p = src[3 * plane + k];
            if (src != dst) {
                dst[o] = rho;
                dst[plane + o] = u;
                dst[2 * plane + o] = v;
                dst[3 * plane + o] = p;
            }
            double t = 0.5 * u * u + p / (gamma - 1.0) / rho;
            t += 0.5 * v * v;
            dst[4 * plane + o] = t;
        } else {
            for (int f = 0; f < nf; ++f) dst[f * plane + o] = src[f * plane + k];
        }
    }
}

// pitched planes to packed ones, the same fields
__global__ void __launch_bounds__(256) pack_kernel(const double *src, double *dst, size_t plane, int m, int n, int ld, int nf)
{
    const size_t total = (size_t)m * n;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (size_t)gridDim.x * blockDim.x) {
        const size_t j = k / n, o = j * ld + (k - j * n);
        for (int f = 0; f < nf; ++f) dst[f * plane + k] = src[f * plane + o];
    }
}

// the BC -1 ghosts from the initial data (bound_cond_slope_limiter_x.c:37-46):
// tables x_lo, x_hi (n x 4), y_lo, y_hi (m x 4), one after the other
__global__ void __launch_bounds__(256) ghost_table_kernel(const double *st, size_t plane, int m, int n, int ld, double *b)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m + n) return;
    const size_t lo = k < n ? (size_t)k : (size_t)(k - n) * ld;
    const size_t hi = k < n ? (size_t)(m - 1) * ld + k : (size_t)(k - n) * ld + (n - 1);
    double *t = k < n ? b + (size_t)k * 4 : b + (size_t)n * 8 + (size_t)(k - n) * 4;
    const size_t far = k < n ? (size_t)n * 4 : (size_t)m * 4;
    for (int q = 0; q < 4; ++q) {
        t[q] = st[q * plane + lo];
        t[far + q] = st[q * plane + hi];
    }
}

// rows that fill their pitch, or a single one: the plane is the packed array
static bool is_packed(int m, int n, int ld) { return n == ld || m == 1; }

static unsigned blocks_of(size_t total)
{
    const size_t b = (total + 255) / 256;
    return (unsigned)(b < 8192 ? b : 8192);
}

hipError_t upload_state(const double *const src[5], double *stage, double *dst, double *bnd, size_t plane, int m, int n,
                        int ld, double gamma, hipStream_t st)
{
    const size_t bytes = (size_t)m * n * 8;
    const int nf = src[4] ? 5 : 4;
    double *to = is_packed(m, n, ld) ? dst : stage;
    for (int f = 0; f < nf; ++f) {
        const hipError_t e = hipMemcpyAsync(to + f * plane, src[f], bytes, hipMemcpyHostToDevice, st);
        if (e != hipSuccess) return e;
    }
    if (to != dst || nf == 4)
        hipLaunchKernelGGL(unpack_kernel, dim3(blocks_of((size_t)m * n)), dim3(256), 0, st, to, dst, plane, m, n, ld, nf,
                           nf == 4, gamma);
    hipLaunchKernelGGL(ghost_table_kernel, dim3((unsigned)((m + n + 255) / 256)), dim3(256), 0, st, dst, plane, m, n, ld,
                       bnd);
    return hipGetLastError();
}

hipError_t upload_plane(const double *src, double *stage, double *dst, int m, int n, int ld, hipStream_t st)
{
    const bool packed = is_packed(m, n, ld);
    const hipError_t e = hipMemcpyAsync(packed ? dst : stage, src, (size_t)m * n * 8, hipMemcpyHostToDevice, st);
    if (e != hipSuccess || packed) return e;
    hipLaunchKernelGGL(unpack_kernel, dim3(blocks_of((size_t)m * n)), dim3(256), 0, st, stage, dst, (size_t)0, m, n, ld, 1,
                       0, 0.0);
    return hipGetLastError();
}

hipError_t download_planes(double *const dst[], int nf, const double *src, double *stage, size_t plane, int m, int n, int ld,
                           hipStream_t st)
{
    // One or two rows come down faster as they lie: a strided copy of one takes 11 us, of two 18, a contiguous one
    // of any small array 16 to 23 (a download of one row 57 us against 79, a fraction's of two 19 against 24)
    if (m == 1 || (m == 2 && nf == 1)) {
        for (int f = 0; f < nf; ++f) {
            if (!dst[f]) continue;
            const hipError_t e = hipMemcpy2DAsync(dst[f], (size_t)n * 8, src + f * plane, (size_t)ld * 8, (size_t)n * 8,
                                                  (size_t)m, hipMemcpyDeviceToHost, st);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    if (n != ld) {
        hipLaunchKernelGGL(pack_kernel, dim3(blocks_of((size_t)m * n)), dim3(256), 0, st, src, stage, plane, m, n, ld, nf);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        src = stage;
    }
    for (int f = 0; f < nf; ++f) {
        if (!dst[f]) continue;
        const hipError_t e = hipMemcpyAsync(dst[f], src + f * plane, (size_t)m * n * 8, hipMemcpyDeviceToHost, st);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace hgrp
