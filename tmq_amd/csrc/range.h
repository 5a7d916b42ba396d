// The power-of-two prescale that brings fp32 values into the range two fp16 terms cover (prescale.hip says why).
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

namespace tmq {

#if defined(__HIPCC__)

__device__ __forceinline__ float finite_abs(float v) {
    const float a = __builtin_fabsf(v);
    return a < INFINITY ? a : 0.f;          // NaN and Inf take no part in the maximum (they propagate anyway)
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// s = 2^(11 - e) for amax in [2^(e-1), 2^e), kept inside the normal range together with its reciprocal.
__device__ __forceinline__ void make_prescale(float amax, float &s, float &inv) {
    s = 1.f;
    inv = 1.f;
    if (!(amax > 0.f)) return;
    int e;
    (void)frexpf(amax, &e);
    int p = 11 - e;
    p = p > 126 ? 126 : (p < -126 ? -126 : p);
    s = ldexpf(1.f, p);
    inv = ldexpf(1.f, -p);
}

#endif

// Launches the scan for the largest finite |x| of n values: partial maxima (at most 1024; the callers' next launch reduces
// them) to `partials`; returns how many. vec: x is 16-byte aligned. (prescale.hip)
int launch_absmax(const float *x, int64_t n, float *partials, int vec, void *stream);

}  // namespace tmq
