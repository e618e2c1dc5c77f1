// The linear-depth rejection |L(hd) - L(d)| > thr, L(x) = n f / (f + x (n - f)) (taa.comp:559-564),
// decided without its two IEEE divisions wherever the rounding cannot matter. Host and device, so
// that the decision is checked on the CPU (tests/test_depth_test.py).
#pragma once

#include <hip/hip_runtime.h>

namespace taastar {

// With q1, q2 the divisors as linearize_depth forms them, the test is |q2 - q1| > k |q1 q2|, k = thr / |n f|.
// Every quotient of the FP32 path is within 2^-24 of its value, so its difference, scaled by |q1 q2| / |n f|,
// is within 2^-24 (|q1| + |q2|) + 2^-23 |q2 - q1| of |q2 - q1|; here k (1 ulp of the hardware reciprocal) and the
// products are within 2^-21. Both together stay below 2^-21 (|q1| + |q2|) + 2^-21 k |q1 q2|: a case farther
// than four times that from the threshold is decided; 1e-20 keeps products that underflow and quotients that
// overflow out. The rest, and every non-finite case, is left to the IEEE divisions.
// Returns 1 (reject), 0 (keep) or -1 (undecided).
__host__ __device__ __forceinline__ int linear_depth_decided(float q1, float q2, float k) {
    const float l = __builtin_fabsf(q2 - q1), r = k * __builtin_fabsf(q1 * q2);
    const float m = __builtin_fmaf(0x1p-19f, r, __builtin_fmaf(0x1p-19f, __builtin_fabsf(q1) + __builtin_fabsf(q2), 1e-20f));
    if (l > r + m) return 1;
    if (l < r - m) return 0;  // a product that overflows leaves inf - inf here
    return -1;
}

}  // namespace taastar
