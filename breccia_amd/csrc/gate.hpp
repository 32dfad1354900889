// The output gate, as every attention kernel applies it.
#pragma once

#include <hip/hip_runtime.h>

namespace bkv {

// sigmoid in the overflow-free form of the reference (qsa/cpu.rs:84-91): 1 / (1 + exp(-x)), below 0 exp(x) / (1 + exp(x)).
// 2^-22 of the result at most: 1 ulp of expf, half of one each for the sum and the quotient.  Subnormal results included
// (x from -87.3 to -104): no bare v_exp_f32, which has none, and no product with a reciprocal.  (Those two: 531 us instead of
// 540 for a prompt of 4096, 24 heads, q8_0 V.  A division without the scaling that a divisor of 1 to 2 does not need, the same
// bits: 540.)
__device__ __forceinline__ float sigmoid(float x) {
    const float ex = expf(-fabsf(x));
    return (x >= 0.0f ? 1.0f : ex) / (1.0f + ex);
}

}  // namespace bkv
