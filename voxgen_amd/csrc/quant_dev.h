// Widening of Q8_0 quants to f16 for the matrix cores (kernels_gemm.hip,
// kernels_prefill_short.hip, kernels_seq.hip).
#pragma once

#include "vx_internal.h"

namespace vx {

// Four quants stored as u = q + 128 (one dword) -> four exact f16 values q: the f16
// with bits 0x6400 | u is 1024 + u, minus 1152 = q.
__device__ __forceinline__ uint2 q8x4_to_f16(uint32_t u) {
    typedef _Float16 h2v __attribute__((ext_vector_type(2)));
    const uint32_t lo = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    const uint32_t hi = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const h2v bias = {(_Float16)1152.0f, (_Float16)1152.0f};
    const h2v a = __builtin_bit_cast(h2v, lo) - bias;
    const h2v b = __builtin_bit_cast(h2v, hi) - bias;
    return make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
}
// Four signed int8 quants: (q ^ 0x80) is q + 128.
__device__ __forceinline__ uint2 q8x4s_to_f16(uint32_t w) { return q8x4_to_f16(w ^ 0x80808080u); }

}  // namespace vx
