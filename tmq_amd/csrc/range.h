// The power-of-two prescale that brings fp32 values into the range two fp16 terms cover (prescale.hip says why).
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

namespace tmq {

#if defined(__HIPCC__)

__device__ __forceinline__ float finite_abs(float v) {
    const float a = __builtin_fabsf(v);
    return a < INFINITY ? a : 0.f;          // NaN and Inf take no part in the maximum (they propagate anyway)
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

}  // namespace tmq
