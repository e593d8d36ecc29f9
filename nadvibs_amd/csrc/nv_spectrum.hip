// Gaussian broadening of stick spectra: the normalised envelope of
// convolve.py:28-48 and the unnormalised one of tridiagonal eigenpairs.
//
// env[g] = sum_j y_j exp(-((grid_g - x_j)/sigma)^2 / 2): ng * n exponentials
// and next to no memory, so the only question is how many waves share them.
// One grid point per thread leaves the chip idle on the usual grids (4096
// points are 16 workgroups: 144 us with 2000 sticks), so up to kSplitGrid
// points kSplit lanes share a point's sticks (23 us); above, a point per thread
// fills the chip and needs no reduction.
#include <hip/hip_runtime.h>

#include "nv_kernels.hpp"

namespace nv {

constexpr int kSplit = 16;             // lanes per grid point
constexpr int64_t kSplitGrid = 65536;  // 4096 workgroups of 16 points, 16 per CU

// 1 / sigma, finite for the subnormal ones too: a stick at the grid point counts in full.
__device__ __forceinline__ double inv_sigma(double sigma) { return fmin(1.0 / sigma, 1.7976931348623157e308); }

// The sum over the sticks at gx; S lanes share it and all return it.  Sticks
// go through LDS in tiles of kBlock; stick(j) gives (position, weight).
template <int S, typename Stick>
__device__ __forceinline__ double gauss_sum(double gx, double inv, int64_t n, Stick stick) {
    __shared__ double sx[kBlock], sy[kBlock];
    double acc = 0.0;
    for (int64_t j0 = 0; j0 < n; j0 += kBlock) {
        __syncthreads();
        if (j0 + threadIdx.x < n) stick(j0 + threadIdx.x, sx[threadIdx.x], sy[threadIdx.x]);
        __syncthreads();
        const int m = (int)(n - j0 < kBlock ? n - j0 : kBlock);
        for (int j = threadIdx.x % S; j < m; j += S) {
            const double t = (gx - sx[j]) * inv;
            acc += sy[j] * exp(-0.5 * t * t);
        }
    }
#pragma unroll
    for (int off = S / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    return acc;
}

template <int S>
__global__ __launch_bounds__(kBlock) void convolve_kernel(const double *x, const double *y, int64_t n,
                                                          const double *grid, int64_t ng, double sigma, double *env,
                                                          double *part) {
    const int64_t g = (int64_t)blockIdx.x * (kBlock / S) + threadIdx.x / S;
    const double acc = gauss_sum<S>(g < ng ? grid[g] : 0.0, inv_sigma(sigma), n, [&](int64_t j, double &sx, double &sy) {
        sx = x[j];
        sy = y[j];
    });
    if (g < ng && threadIdx.x % S == 0) env[g] = acc;
    // block maximum for the normalisation
    double mx = g < ng ? acc : -INFINITY;
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    __shared__ double red[kBlock / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m2 = red[0];
        for (int w = 1; w < kBlock / 64; ++w) m2 = fmax(m2, red[w]);
        part[blockIdx.x] = m2;
    }
}

__global__ __launch_bounds__(kBlock) void convolve_norm_kernel(double *env, int64_t ng, const double *part, int nb) {
    __shared__ double red[kBlock / 64];
    double mx = -INFINITY;
    for (int b = threadIdx.x; b < nb; b += kBlock) mx = fmax(mx, part[b]);
    for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    for (int w = 0; w < kBlock / 64; ++w) mx = fmax(mx, red[w]);
    for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < ng; g += (int64_t)gridDim.x * kBlock)
        env[g] /= mx;
}

int64_t convolve_parts(int64_t ng) {
    const int64_t per = ng <= kSplitGrid ? kBlock / kSplit : kBlock;
    return (ng + per - 1) / per;
}

hipError_t launch_convolve(const double *x, const double *y, int64_t n, const double *grid, int64_t ng,
                           double sigma, double *env, double *part, hipStream_t s) {
    const int np = (int)convolve_parts(ng);
    if (ng <= kSplitGrid)
        hipLaunchKernelGGL(convolve_kernel<kSplit>, dim3(np), dim3(kBlock), 0, s, x, y, n, grid, ng, sigma, env,
                           part);
    else
        hipLaunchKernelGGL(convolve_kernel<1>, dim3(np), dim3(kBlock), 0, s, x, y, n, grid, ng, sigma, env, part);
    hipLaunchKernelGGL(convolve_norm_kernel, dim3((unsigned)((ng + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, env,
                       ng, part, np);
    return hipGetLastError();
}

// ---- broadened spectrum of the tridiagonal eigenpairs -------------------------
// env[g] = sum_i a_i^2 G(grid[g] - (theta_i - ref) c),  a_i = vec[i] (first
// components), G(u) = exp(-u^2 / (2 sigma^2)).
template <int S>
__global__ __launch_bounds__(kBlock) void spec_env_kernel(int64_t n, const double *__restrict__ theta,
                                                         const double *__restrict__ vec, double ref, double c,
                                                         double sigma, int64_t ng, const double *__restrict__ grid,
                                                         double *__restrict__ env) {
    const int64_t g = (int64_t)blockIdx.x * (kBlock / S) + threadIdx.x / S;
    const double acc = gauss_sum<S>(g < ng ? grid[g] : 0.0, inv_sigma(sigma), n, [&](int64_t i, double &sx, double &sy) {
        const double a = vec[i];
        sx = (theta[i] - ref) * c;
        sy = a * a;
    });
    if (g < ng && threadIdx.x % S == 0) env[g] = acc;
}

hipError_t launch_spec_env(int64_t n, const double *theta, const double *vec, double ref, double c, double sigma,
                           int64_t ng, const double *grid, double *env, hipStream_t s) {
    const unsigned nb = (unsigned)convolve_parts(ng);
    if (ng <= kSplitGrid)
        hipLaunchKernelGGL(spec_env_kernel<kSplit>, dim3(nb), dim3(kBlock), 0, s, n, theta, vec, ref, c, sigma, ng,
                           grid, env);
    else
        hipLaunchKernelGGL(spec_env_kernel<1>, dim3(nb), dim3(kBlock), 0, s, n, theta, vec, ref, c, sigma, ng, grid,
                           env);
    return hipGetLastError();
}

}  // namespace nv
