/* Device helpers of the output RMS norm (cpu_scalar_rmsnorm,
 * src/backends/cpu_scalar/elementwise.c:241-280), shared by the kernels that norm a hidden row. */
#ifndef GEIST_RMSNORM_DEVICE_H
#define GEIST_RMSNORM_DEVICE_H

#include <hip/hip_runtime.h>

namespace gs {

/* 1 / sqrt(mean(x^2) + eps) as cpu_scalar_rmsnorm rounds it (elementwise.c:270-274). The
 * reference adds the squares in double in index order; the order of a double sum only shows in
 * the binary32 result when the value lies within the sums' error of the middle between two
 * binary32 values, and then `sequential` repeats the sum in the reference's order. */
__device__ __forceinline__ bool rms_inv_is_safe(double sumsq, int n, float eps, float &f) {
    const double r  = 1.0 / sqrt(sumsq / (double) n + (double) eps);
    f               = (float) r;
    const float  fn = r > (double) f ? nextafterf(f, __builtin_inff()) : nextafterf(f, -__builtin_inff());
    const double mid = 0.5 * ((double) f + (double) fn);
    return !(fabs(r - mid) <= fabs(r) * (double) n * 0x1p-50);
}
__device__ __forceinline__ float rms_inv_sequential(const float *__restrict__ xr, int n, float eps) {
    double sumsq = 0.0;
    for (int i = 0; i < n; ++i)
        sumsq += (double) xr[i] * (double) xr[i];
    return (float) (1.0 / sqrt(sumsq / (double) n + (double) eps));
}

/* The threads that norm one row where there are few rows. One row is one workgroup's work, and it is
 * latency that it takes: the row's and the weights' elements are asked for at once, four of each per
 * thread, and stay in registers. 256 threads that looped over memory twice, and added their sums
 * through LDS in eight barriers, took 11.2 us of a cold step for the norm of 2560 elements where this
 * takes 5.3 (4.6 is what any launch takes), with the Q6_K quantiser 11.5 against 5.8, with the Q4_K
 * one for 8 rows of 1536 9.5 against 5.5, with the sketch head's activations 13.8 against 6.0. */
constexpr int NORM_TPB = 1024;
constexpr int NORM_PER = 4;

struct NormShared {
    double part[NORM_TPB / 64];
    float  inv;
};

/* The inverse RMS of xr[0..n) for a workgroup of TPB threads, every thread gets it, and in
 * v[k] the normed element (x inv) w at k TPB + tid (0 from n on); elements from PER TPB on are the
 * caller's. The squares are added in double in a fixed parallel order
 * (a thread's elements ascending, then a butterfly over the lanes and over the wavefronts) and,
 * where the binary32 result could depend on the order, once more by one thread in the reference's
 * order. One call per launch (s is not given free for another). */
template <int TPB = NORM_TPB, int PER = NORM_PER>
__device__ __forceinline__ float block_rmsnorm(const float *__restrict__ xr,
                                               const float *__restrict__ w, int n, float eps,
                                               float (&v)[PER], NormShared &s) {
    const int tid = threadIdx.x;
    float     wv[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int i = k * TPB + tid;
        v[k]        = i < n ? xr[i] : 0.0f;
        wv[k]       = i < n ? w[i] : 0.0f;
    }
    double a = 0.0;
#pragma unroll
    for (int k = 0; k < PER; ++k)
        a += (double) v[k] * (double) v[k];
    for (int i = PER * TPB + tid; i < n; i += TPB)
        a += (double) xr[i] * (double) xr[i];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        a += __shfl_xor(a, d);
    if ((tid & 63) == 0)
        s.part[tid >> 6] = a;
    __syncthreads();
    if (tid < 64) {
        a = s.part[tid & (TPB / 64 - 1)];
#pragma unroll
        for (int d = TPB / 128; d >= 1; d >>= 1)
            a += __shfl_xor(a, d);
        if (tid == 0) {
            float f;
            if (!rms_inv_is_safe(a, n, eps, f))
                f = rms_inv_sequential(xr, n, eps);
            s.inv = f;
        }
    }
    __syncthreads();
    const float inv = s.inv;
#pragma unroll
    for (int k = 0; k < PER; ++k)
        v[k] = __fmul_rn(__fmul_rn(v[k], inv), wv[k]);
    return inv;
}

/* The largest of the threads' values (a NaN is passed over); s: NORM_TPB / 64 floats. */
__device__ __forceinline__ float block_norm_max(float ax, float *s) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        ax = __builtin_fmaxf(ax, __shfl_xor(ax, d));
    if ((threadIdx.x & 63) == 0)
        s[threadIdx.x >> 6] = ax;
    __syncthreads();
    ax = s[threadIdx.x & (NORM_TPB / 64 - 1)];
#pragma unroll
    for (int d = NORM_TPB / 128; d >= 1; d >>= 1)
        ax = __builtin_fmaxf(ax, __shfl_xor(ax, d));
    return ax;
}

} // namespace gs
#endif
