/* When a double sum formed in another order than the reference's rounds to the reference's binary32
 * all the same. */
#ifndef GEIST_F32_ROUNDING_H
#define GEIST_F32_ROUNDING_H

#include <hip/hip_runtime.h>

namespace gs {

/* (float) s for a finite s, and whether every value within err of s rounds to the same binary32:
 * s lies closer to it than half a step by more than err. (At a power of two the step below is
 * half of the one above: taken for both. 2^128 stands for infinity, which begins half a step below
 * it. The bounds passed as err have room for the rounding of the sum here.) */
__device__ __forceinline__ bool f32_rounding_is_safe(double s, double err, float &f) {
    const double    a = fmin(fabs(s), 0x1p128);
    const float     g = (float) a;
    const double    v = fmin((double) g, 0x1p128);
    const long long b = __double_as_longlong(v), exponent = 0x7ffll << 52;
    const double    half = __longlong_as_double(b & exponent) * ((b & ~exponent) ? 0x1p-24 : 0x1p-25);
    f = copysignf(g, (float) s);
    return fabs(a - v) + err < fmax(half, 0x1p-150);
}

} // namespace gs
#endif
