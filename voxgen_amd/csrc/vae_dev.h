// Device helpers shared by the AudioVAE decode kernels (kernels_vae.hip,
// kernels_vae_unit.hip).
#pragma once

#include "vx_internal.h"

namespace vx {

// sin(v)^2 for |v| < kSinSqMax. Cody-Waite reduction to r = v - n pi/2 in
// [-pi/4, pi/4] (pi/2 as a sum of two floats, fused multiply-adds), then
// sin(r)^2 = z + z^2 P(z), z = r^2, with P the polynomial of least largest relative
// error on z <= 1.01 (pi/4)^2 (9.5e-10; fitted by Lawson's iteration on the Taylor
// series of sin^2), and sin(v)^2 = 1 - sin(r)^2 for odd n. Against 64 bits on
// N(0, 1..1e4): rms error 1.9e-8 (a rounded sine squared: 2.7e-8), largest 1.0e-7.
// 14 instructions, where sinf takes about 40 with the branch for large arguments.
constexpr float kSinSqMax = 32768.0f;
__device__ __forceinline__ float sin_sq(float v) {
    constexpr float kRound = 12582912.0f;   // 1.5 * 2^23: adding it leaves n in the low bits
    const float m = fmaf(v, 0.63661975f, kRound), n = m - kRound;
    float r = fmaf(-n, 1.57079637f, v);
    r = fmaf(-n, -4.37113883e-8f, r);
    const float z = r * r;
    float p = fmaf(1.34681002e-4f, z, -3.17122882e-3f);
    p = fmaf(p, z, 4.44437390e-2f);
    p = fmaf(p, z, -3.33333287e-1f);
    const float t = fmaf(p, z * z, z);
    return (__builtin_bit_cast(uint32_t, m) & 1u) ? 1.0f - t : t;
}
// Any argument (the caller's rare path).
__device__ __forceinline__ float sin_sq_any(float v) {
    const float s = sinf(v);
    return s * s;
}

__device__ __forceinline__ float vae_h2f(__half v) { return __half2float(v); }

// The snake's 1 / (a + 1e-9), computed once per channel.
__device__ __forceinline__ float snake_inv(float a) { return 1.0f / (a + 1e-9f); }

// Whether any lane of the wave has an argument outside sin_sq's range.
__device__ __forceinline__ bool any_large(float big) { return __any(!(big < kSinSqMax)) != 0; }

}  // namespace vx
