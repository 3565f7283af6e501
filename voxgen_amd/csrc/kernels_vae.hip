// AudioVAE decoder kernels (vae_*.comp).
//
// Two families:
//  * channel-major [C][L] kernels with the reference shaders' semantics, behind
//    the per-op entry points (vae_conv1d.comp, vae_convtranspose1d.comp,
//    vae_snake.comp, vae_scale_bias.comp, vae_add.comp, vae_tanh.comp);
//  * frame-major [L][C] kernels of the decode engine, where the 1x1 convolutions
//    and the transposed convolutions are GEMMs on MFMA (k_gemm) and the
//    elementwise work (scale/bias, snake) is fused into the passes around them.
// Snake: x + sin(a x)^2 / (a + 1e-9) (vae_snake.comp:13-16).
#include "vae_dev.h"

namespace vx {
namespace {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));


__device__ __forceinline__ float hf(__half v) { return __half2float(v); }

// A model scalar of GGML dtype 1 (F16) or 0 (F32).
__device__ __forceinline__ float ldw(const void *p, uint32_t i, uint32_t dtype) {
    return dtype == 1u ? hf(static_cast<const __half *>(p)[i]) : static_cast<const float *>(p)[i];
}

__device__ __forceinline__ float snake(float x, float a) {
    const float s = sinf(a * x);
    return x + (s * s) / (a + 1e-9f);
}
// The decode engine's snake with the channel's 1 / (a + 1e-9) computed once:
// x + sin(ax)^2 inv, ax = a x inside sin_sq's range.
__device__ __forceinline__ float snake_fm(float x, float ax, float inv) { return fmaf(sin_sq(ax), inv, x); }
__device__ __forceinline__ float snake_any(float x, float ax, float inv) { return fmaf(sin_sq_any(ax), inv, x); }

// Lane exchanges inside a row of 16 lanes (gfx9 DPP controls).
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
// Sum over each 8 consecutive lanes: quad swaps, then the half-row mirror.
__device__ __forceinline__ float sum8(float v) {
    v += dpp<0xb1>(v);   // quad_perm [1,0,3,2]
    v += dpp<0x4e>(v);   // quad_perm [2,3,0,1]
    return v + dpp<0x141>(v);   // row_half_mirror
}

// ------------------------------------------------------------ channel-major
__global__ __launch_bounds__(256) void k_vae_conv1d_cm(VaeConvArgs a) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, oc = blockIdx.y;
    if (t >= a.out_length || oc >= a.out_channels) return;
    const uint32_t out_pg = a.out_channels / a.groups, in_pg = a.in_channels / a.groups;
    const uint32_t in_base = (oc / out_pg) * in_pg;
    float sum = a.bias ? ldw(a.bias, oc, a.bias_dtype) : 0.f;
    for (uint32_t icg = 0; icg < in_pg; ++icg) {
        const uint32_t ic = in_base + icg;
        for (uint32_t k = 0; k < a.kernel; ++k) {
            const int ti = (int)(t * a.stride + k * a.dilation) - (int)a.left_pad;
            if (ti < 0 || ti >= (int)a.in_length) continue;
            const float w = ldw(a.w, (oc * in_pg + icg) * a.kernel + k, a.w_dtype);
            sum += a.x[(size_t)ic * a.in_length + (uint32_t)ti] * w;
        }
    }
    a.y[(size_t)oc * a.out_length + t] = sum;
}

__global__ __launch_bounds__(256) void k_vae_convt1d_cm(VaeConvArgs a) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, oc = blockIdx.y;
    if (t >= a.out_length || oc >= a.out_channels) return;
    const uint32_t out_pg = a.out_channels / a.groups, in_pg = a.in_channels / a.groups;
    const uint32_t group = oc / out_pg, ocg = oc - group * out_pg, in_base = group * in_pg;
    float sum = a.bias ? ldw(a.bias, oc, a.bias_dtype) : 0.f;
    const uint32_t first_k = t % a.stride;
    for (uint32_t icg = 0; icg < in_pg; ++icg) {
        const uint32_t ic = in_base + icg;
        for (uint32_t k = first_k; k < a.kernel; k += a.stride) {
            if (t < k) continue;
            const uint32_t ti = (t - k) / a.stride;
            if (ti >= a.in_length) continue;
            sum += a.x[(size_t)ic * a.in_length + ti] * ldw(a.w, (ic * out_pg + ocg) * a.kernel + k, a.w_dtype);
        }
    }
    a.y[(size_t)oc * a.out_length + t] = sum;
}

__global__ __launch_bounds__(256) void k_vae_snake_cm(const float *x, float *y, const void *alpha, uint32_t dtype,
                                                      uint32_t channels, uint32_t length) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, c = blockIdx.y;
    if (t >= length || c >= channels) return;
    const size_t i = (size_t)c * length + t;
    y[i] = snake(x[i], ldw(alpha, c, dtype));
}

__global__ __launch_bounds__(256) void k_vae_scale_bias_cm(float *x, const void *scale, const void *bias,
                                                           uint32_t sdt, uint32_t bdt, uint32_t channels,
                                                           uint32_t length, uint32_t bucket) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, c = blockIdx.y;
    if (t >= length || c >= channels) return;
    const size_t i = (size_t)c * length + t;
    const uint32_t idx = bucket * channels + c;
    x[i] = x[i] * ldw(scale, idx, sdt) + ldw(bias, idx, bdt);
}

__global__ __launch_bounds__(256) void k_vae_add_cm(float *a, const float *b, uint32_t channels, uint32_t length) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, c = blockIdx.y;
    if (t >= length || c >= channels) return;
    const size_t i = (size_t)c * length + t;
    a[i] += b[i];
}

__global__ __launch_bounds__(256) void k_vae_tanh(float *x, uint32_t n) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) x[i] = tanhf(x[i]);
}

// -------------------------------------------------------------- frame-major
// Depthwise k-tap convolution over [L][C] rows, stride 1, dilation d, left pad
// (causal): y[t][c] = post(b[c] + sum_k w[c][k] pre(x[t + k d - pad][c])), where
// pre / post are the snake of alpha_in / alpha_out when given. One thread per
// (t, c), c fastest.
__global__ __launch_bounds__(256) void k_vae_dwconv_fm(VaeDwArgs a) {
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= (uint64_t)a.length * a.channels) return;
    const uint32_t t = (uint32_t)(i / a.channels), c = (uint32_t)(i - (uint64_t)t * a.channels);
    const float ain = a.alpha_in ? hf(a.alpha_in[c]) : 0.f;
    float sum = hf(a.b[c]);
    for (uint32_t k = 0; k < a.kernel; ++k) {
        const int ti = (int)(t + k * a.dilation) - (int)a.left_pad;
        if (ti < 0) continue;
        float v = a.x[(size_t)ti * a.channels + c];
        if (a.alpha_in) v = snake(v, ain);
        sum += v * hf(a.w[c * a.kernel + k]);
    }
    if (a.alpha_out) sum = snake(sum, hf(a.alpha_out[c]));
    a.y[i] = sum;
}

// The same convolution when left_pad = (kernel - 1) * dilation (the causal
// layers) and kernel <= KMAX, tiled: a workgroup covers TB = 2048 / CB rows of CB
// channels (CB a power of two <= 64, so each thread keeps one channel), stages
// pre(x) for its rows and their left halo in LDS once (pre(0) = 0, so the zero
// padding stays zero), then takes the taps from LDS with the channel's weights,
// bias and snake alphas in registers. Every staging load is issued before the
// first is used.
template <int KMAX>
__global__ __launch_bounds__(256) void k_vae_dwconv_tiled_fm(VaeDwArgs a, uint32_t cb_shift) {
    constexpr uint32_t kMaxHalo = 54u, NS = (2048u + 64u * kMaxHalo + 255u) / 256u;
    __shared__ float xs[2048 + 64 * kMaxHalo];
    const uint32_t CB = 1u << cb_shift, TB = 2048u >> cb_shift, halo = a.left_pad;
    const uint32_t t0 = blockIdx.x * TB, C = a.channels, tid = threadIdx.x;
    const uint32_t cc = tid & (CB - 1u), c = blockIdx.y * CB + cc;
    const bool cval = c < C;
    const uint32_t n_st = (TB + halo) << cb_shift;
    float xv[NS];
#pragma unroll
    for (uint32_t i = 0; i < NS; ++i) {
        const uint32_t idx = tid + 256u * i;
        const int ti = (int)(t0 + (idx >> cb_shift)) - (int)halo;
        xv[i] = idx < n_st && cval && ti >= 0 && (uint32_t)ti < a.length ? a.x[(size_t)ti * C + c] : 0.f;
    }
    const float ain = a.alpha_in && cval ? hf(a.alpha_in[c]) : 0.f;
    const float aout = a.alpha_out && cval ? hf(a.alpha_out[c]) : 0.f;
    const float iin = snake_inv(ain), iout = snake_inv(aout);
    const float bias = cval ? hf(a.b[c]) : 0.f;
    float wk[KMAX];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) wk[k] = cval && (uint32_t)k < a.kernel ? hf(a.w[c * a.kernel + k]) : 0.f;
    float big = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < NS; ++i) {
        const uint32_t idx = tid + 256u * i;
        big = fmaxf(big, fabsf(ain * xv[i]));
        if (idx < n_st) xs[idx] = a.alpha_in ? snake_fm(xv[i], ain * xv[i], iin) : xv[i];
    }
    if (a.alpha_in && any_large(big)) {
#pragma unroll 1
        for (uint32_t idx = tid; idx < n_st; idx += 256u) {
            const int ti = (int)(t0 + (idx >> cb_shift)) - (int)halo;
            if (!cval || ti < 0 || (uint32_t)ti >= a.length) continue;
            const float v = a.x[(size_t)ti * C + c];
            xs[idx] = snake_any(v, ain * v, iin);
        }
    }
    __syncthreads();
    auto conv = [&](uint32_t r) {
        float sum = bias;
#pragma unroll
        for (int k = 0; k < KMAX; ++k)
            if ((uint32_t)k < a.kernel) sum += xs[((r + k * a.dilation) << cb_shift) + cc] * wk[k];
        return sum;
    };
    auto put = [&](uint32_t t, float v) {
        if (!a.yh) {
            a.y[(size_t)t * C + c] = v;
            return;
        }
        const size_t o = tiled_plane_index(t, c, C);
        const _Float16 h = (_Float16)v;
        a.yh[o] = __builtin_bit_cast(__half, h);
        a.yl[o] = __builtin_bit_cast(__half, (_Float16)(v - (float)h));
    };
    big = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < 8u; ++i) {   // TB * CB = 2048 outputs, 8 per thread
        const uint32_t r = (tid + 256u * i) >> cb_shift, t = t0 + r;
        if (t >= a.length || !cval) continue;
        const float sum = conv(r);
        big = fmaxf(big, fabsf(aout * sum));
        put(t, a.alpha_out ? snake_fm(sum, aout * sum, iout) : sum);
    }
    if (a.alpha_out && any_large(big)) {
#pragma unroll 1
        for (uint32_t i = 0; i < 8u; ++i) {
            const uint32_t r = (tid + 256u * i) >> cb_shift, t = t0 + r;
            if (t >= a.length || !cval) continue;
            const float sum = conv(r);
            put(t, snake_any(sum, aout * sum, iout));
        }
    }
}

// Seven taps over few rows: a thread computes two neighbouring channels of one row
// straight from the input, all loads issued before the first is used. Against the tiled
// kernel this takes the snake of every input up to seven times, but has a thread for
// every pair of outputs, no LDS and no barrier (32 rows of 1024 channels are 16 tiled
// workgroups: 8.8 -> 4.3 us). Below 1.5 M outputs only: the snakes are then under 4 us of
// the chip.
__global__ __launch_bounds__(256) void k_vae_dw7_fm(VaeDwArgs a) {
    const uint32_t i = 2u * (blockIdx.x * 256u + threadIdx.x), C = a.channels;
    if (i >= a.length * C) return;
    const uint32_t t = i / C, c = i - t * C;
    float2 x[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        const int r = (int)(t + (uint32_t)k * a.dilation) - (int)a.left_pad;
        x[k] = r >= 0 ? *reinterpret_cast<const float2 *>(a.x + (size_t)r * C + c) : make_float2(0.f, 0.f);
    }
    float w[2][7], sum[2], ai[2] = {0.f, 0.f}, ao[2] = {0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int k = 0; k < 7; ++k) w[j][k] = hf(a.w[(c + j) * 7u + k]);
        sum[j] = hf(a.b[c + j]);
        if (a.alpha_in) ai[j] = hf(a.alpha_in[c + j]);
        if (a.alpha_out) ao[j] = hf(a.alpha_out[c + j]);
    }
    float big = 0.f;
    if (a.alpha_in) {
        const float inv0 = snake_inv(ai[0]), inv1 = snake_inv(ai[1]);
#pragma unroll
        for (int k = 0; k < 7; ++k) {   // snake(0) = 0: the padding stays zero
            const float s0 = ai[0] * x[k].x, s1 = ai[1] * x[k].y;
            big = fmaxf(big, fmaxf(fabsf(s0), fabsf(s1)));
            x[k] = make_float2(snake_fm(x[k].x, s0, inv0), snake_fm(x[k].y, s1, inv1));
        }
        if (any_large(big)) {
#pragma unroll
            for (int k = 0; k < 7; ++k) {
                const int r = (int)(t + (uint32_t)k * a.dilation) - (int)a.left_pad;
                if (r < 0) continue;
                const float2 v = *reinterpret_cast<const float2 *>(a.x + (size_t)r * C + c);
                x[k] = make_float2(snake_any(v.x, ai[0] * v.x, inv0), snake_any(v.y, ai[1] * v.y, inv1));
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        sum[0] += x[k].x * w[0][k];
        sum[1] += x[k].y * w[1][k];
    }
    if (a.alpha_out) {
        const bool large = any_large(fmaxf(fabsf(ao[0] * sum[0]), fabsf(ao[1] * sum[1])));
#pragma unroll
        for (int j = 0; j < 2; ++j)
            sum[j] = large ? snake_any(sum[j], ao[j] * sum[j], snake_inv(ao[j]))
                           : snake_fm(sum[j], ao[j] * sum[j], snake_inv(ao[j]));
    }
    if (!a.yh) {
        *reinterpret_cast<float2 *>(a.y + i) = make_float2(sum[0], sum[1]);
        return;
    }
    const size_t o = tiled_plane_index(t, c, C);
    const h2v hv = {(_Float16)sum[0], (_Float16)sum[1]};
    const h2v lv = {(_Float16)(sum[0] - (float)hv[0]), (_Float16)(sum[1] - (float)hv[1])};
    *reinterpret_cast<h2v *>(a.yh + o) = hv;
    *reinterpret_cast<h2v *>(a.yl + o) = lv;
}

// The input of a stage's transposed convolution, P = snake_pa(x * ps + pt) per
// channel (pre: f32 [4][C]: ps, pt, pa, 1 / (pa + 1e-9)). P is kept with a zero row
// ahead of row 0: the GEMM row of output time j is [P[j-1] | P[j]], which is
// contiguous there, so the rows overlap and nothing is copied twice.
template <int V>
__global__ __launch_bounds__(256) void k_vae_pre_fm(const float *x, float *y, const float *pre, uint32_t C,
                                                    uint64_t n) {
    const uint64_t i = ((uint64_t)blockIdx.x * 256u + threadIdx.x) * V;
    if (i >= n) return;
    const uint32_t c = (uint32_t)(i % C);
    float v[V], s[V], big = 0.f;
    if constexpr (V == 4) {
        const float4 q = *reinterpret_cast<const float4 *>(x + i);
        v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
    } else {
        v[0] = x[i];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
        v[j] = fmaf(v[j], pre[c + j], pre[C + c + j]);
        s[j] = pre[2u * C + c + j] * v[j];
        big = fmaxf(big, fabsf(s[j]));
    }
    if (any_large(big)) {
#pragma unroll 1
        for (int j = 0; j < V; ++j) {
            const float w = fmaf(x[i + j], pre[c + j], pre[C + c + j]);
            y[i + j] = snake_any(w, pre[2u * C + c + j] * w, pre[3u * C + c + j]);
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = snake_fm(v[j], s[j], pre[3u * C + c + j]);
    if constexpr (V == 4)
        *reinterpret_cast<float4 *>(y + i) = make_float4(v[0], v[1], v[2], v[3]);
    else
        y[i] = v[0];
}

// P as block-major planes: one thread per eight channels of a row, the threads of a
// 32-channel block consecutive, so that a wave reads 128-byte runs and writes one of
// 1 KB a plane (row by row, with 64-byte runs: 20 us at 2016 x 1024, this way 5.5); the
// threads of row 0 also zero row -1.
__global__ __launch_bounds__(256) void k_vae_pre_planes(const float *x, VaePlanes y, const float *pre, uint32_t C,
                                                        uint32_t length) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, t = i >> 2, c = blockIdx.y * 32u + 8u * (i & 3u);
    if (t >= length) return;
    float v[8], s[8], inv[8], big = 0.f;
    const float *const xr = x + (size_t)t * C + c;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const float4 q = *reinterpret_cast<const float4 *>(xr + 4 * h);
        const float4 p[4] = {*reinterpret_cast<const float4 *>(pre + c + 4 * h),
                             *reinterpret_cast<const float4 *>(pre + C + c + 4 * h),
                             *reinterpret_cast<const float4 *>(pre + 2u * C + c + 4 * h),
                             *reinterpret_cast<const float4 *>(pre + 3u * C + c + 4 * h)};
        const float qv[4] = {q.x, q.y, q.z, q.w}, ps[4] = {p[0].x, p[0].y, p[0].z, p[0].w},
                    pt[4] = {p[1].x, p[1].y, p[1].z, p[1].w}, pa[4] = {p[2].x, p[2].y, p[2].z, p[2].w},
                    pi[4] = {p[3].x, p[3].y, p[3].z, p[3].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[4 * h + j] = fmaf(qv[j], ps[j], pt[j]);
            s[4 * h + j] = pa[j] * v[4 * h + j];
            inv[4 * h + j] = pi[j];
            big = fmaxf(big, fabsf(s[4 * h + j]));
        }
    }
    __half *const yh = y.h + (size_t)blockIdx.y * (y.block / 2u), *const yl = y.l + (size_t)blockIdx.y * (y.block / 2u);
    const size_t o = (size_t)t * 32u + 8u * ((i & 3u) ^ xperm(t));
    if (t == 0u) {
        *reinterpret_cast<h8v *>(yh + 8u * (i & 3u) - 32) = h8v{};
        *reinterpret_cast<h8v *>(yl + 8u * (i & 3u) - 32) = h8v{};
    }
    if (any_large(big)) {
#pragma unroll 1
        for (uint32_t j = 0; j < 8u; ++j) {
            const float w = fmaf(xr[j], pre[c + j], pre[C + c + j]);
            const float r = snake_any(w, pre[2u * C + c + j] * w, pre[3u * C + c + j]);
            const _Float16 h = (_Float16)r;
            yh[o + j] = __builtin_bit_cast(__half, h);
            yl[o + j] = __builtin_bit_cast(__half, (_Float16)(r - (float)h));
        }
        return;
    }
    h8v hv, lv;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float r = snake_fm(v[j], s[j], inv[j]);
        hv[j] = (_Float16)r;
        lv[j] = (_Float16)(r - (float)hv[j]);
    }
    *reinterpret_cast<h8v *>(yh + o) = hv;
    *reinterpret_cast<h8v *>(yl + o) = lv;
}

__global__ __launch_bounds__(256) void k_vae_repack_pre(const __half *scale, const __half *bias, const __half *alpha,
                                                        uint32_t C, float *pre) {
    const uint32_t c = blockIdx.x * 256u + threadIdx.x;
    if (c >= C) return;
    pre[c] = hf(scale[c]);
    pre[C + c] = hf(bias[c]);
    pre[2u * C + c] = hf(alpha[c]);
    pre[3u * C + c] = snake_inv(hf(alpha[c]));
}

// Repack of a ConvTranspose1d weight [Cin][Cout][2s] (kernel 2s, stride s) for
// the GEMM form: W'[(r Cout + oc)][(1 - tap) Cin + ic] = W[ic][oc][r + tap s] (tap 1
// multiplies the earlier row, which comes first), and the bias tiled over the s phases, b'[r Cout + oc] = b[oc].
__global__ __launch_bounds__(256) void k_vae_repack_convt(const __half *w, const __half *b, uint32_t cin,
                                                          uint32_t cout, uint32_t s, uint32_t prefill_layout,
                                                          __half *wp, float *bp) {
    const uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    const uint64_t n = (uint64_t)s * cout * 2u * cin;
    if (i < n) {
        const uint32_t row = (uint32_t)(i / (2u * cin)), col = (uint32_t)(i - (uint64_t)row * 2u * cin);
        const uint32_t r = row / cout, oc = row - r * cout, tap = col / cin, ic = col - tap * cin;
        wp[prefill_layout ? tiled_plane_index(row, col, 2u * cin) : i] =
            w[((size_t)ic * cout + oc) * (2u * s) + r + (1u - tap) * s];
    } else if (prefill_layout && i < (uint64_t)((s * cout + 127u) / 128u * 128u) * 2u * cin) {   // padding rows
        wp[tiled_plane_index((uint32_t)(i / (2u * cin)), (uint32_t)(i % (2u * cin)), 2u * cin)] = __float2half(0.f);
    }
    if (i < (uint64_t)s * cout) bp[i] = hf(b[i % cout]);
}

// y[t][n] (+)= b[n] + sum_k x[t][k] W[n][k] for short K (the GEMM takes K % 128
// == 0): a workgroup covers NB = min(N, 256) outputs of RB rows, the rows staged
// in LDS; thread (g, n) computes rows g, g + G, ... (G = 256 / NB, at most
// kLinRows of them) together, reading W[n] once in 8-column chunks (K % 8 == 0). Rows past
// a short batch are left out: 8.4 -> 6.0 us for the decoder's stem at 4 frames.
constexpr uint32_t kLinRows = 8;
__global__ __launch_bounds__(256) void k_vae_linear_fm(VaeLinearArgs a, uint32_t NB, uint32_t RB) {
    extern __shared__ float xs[];
    const uint32_t tid = threadIdx.x, G = 256u / NB, n = blockIdx.x * NB + tid % NB, g = tid / NB;
    const uint32_t r0 = blockIdx.y * RB;
    for (uint32_t idx = tid; idx < RB * a.K; idx += 256u) {
        const uint32_t r = idx / a.K, k = idx - r * a.K;
        xs[idx] = r0 + r < a.T ? a.x[(size_t)(r0 + r) * a.ldx + k] : 0.f;
    }
    __syncthreads();
    if (n >= a.N || g >= G) return;
    const __half *w = a.w + (size_t)n * a.K;
    const float b = a.bias_f32 ? a.bias_f32[n] : (a.bias ? hf(a.bias[n]) : 0.f);
    float acc[kLinRows];
#pragma unroll
    for (uint32_t j = 0; j < kLinRows; ++j) acc[j] = 0.f;
    for (uint32_t k0 = 0; k0 < a.K; k0 += 8u) {
        const uint4 wc = *reinterpret_cast<const uint4 *>(w + k0);
        const uint32_t wu[4] = {wc.x, wc.y, wc.z, wc.w};
        float wf[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const __half2 h = __builtin_bit_cast(__half2, wu[e]);
            wf[2 * e] = __low2float(h);
            wf[2 * e + 1] = __high2float(h);
        }
#pragma unroll
        for (uint32_t j = 0; j < kLinRows; ++j) {
            const uint32_t r = g + G * j;
            if (r >= RB || r0 + r >= a.T) break;
            const float *xr = xs + r * a.K + k0;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[j] += xr[e] * wf[e];
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < kLinRows; ++j) {
        const uint32_t r = g + G * j;
        if (r >= RB || r0 + r >= a.T) break;
        const float v = acc[j] + b;
        float *dst = a.y + (size_t)(r0 + r) * a.ldy + n;
        *dst = a.residual ? *dst + v : v;
    }
}

// Any K and weight alignment: W[n][k] read element by element.
__global__ __launch_bounds__(256) void k_vae_linear_fm_any(VaeLinearArgs a, uint32_t NB, uint32_t RB) {
    extern __shared__ float xs[];
    const uint32_t tid = threadIdx.x, G = 256u / NB, n = blockIdx.x * NB + tid % NB, g = tid / NB;
    const uint32_t r0 = blockIdx.y * RB;
    for (uint32_t idx = tid; idx < RB * a.K; idx += 256u) {
        const uint32_t r = idx / a.K, k = idx - r * a.K;
        xs[idx] = r0 + r < a.T ? a.x[(size_t)(r0 + r) * a.ldx + k] : 0.f;
    }
    __syncthreads();
    if (n >= a.N || g >= G) return;
    const __half *w = a.w + (size_t)n * a.K;
    const float b = a.bias_f32 ? a.bias_f32[n] : (a.bias ? hf(a.bias[n]) : 0.f);
    for (uint32_t r = g; r < RB && r0 + r < a.T; r += G) {
        float sum = 0.f;
        for (uint32_t k = 0; k < a.K; ++k) sum += xs[r * a.K + k] * hf(w[k]);
        const float v = sum + b;
        float *dst = a.y + (size_t)(r0 + r) * a.ldy + n;
        *dst = a.residual ? *dst + v : v;
    }
}

// Decoder head: wave[t] = tanh(b + sum_c sum_k w[c][k] snake(x[t + k - pad][c])),
// one output channel (model.8 snake, model.9 conv, vae_tanh.comp).
__global__ __launch_bounds__(256) void k_vae_head_fm(VaeHeadArgs a) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= a.length) return;
    float sum = hf(a.b[0]);
    for (uint32_t c = 0; c < a.channels; ++c) {
        const float al = hf(a.alpha[c]);
        for (uint32_t k = 0; k < a.kernel; ++k) {
            const int ti = (int)(t + k) - (int)a.left_pad;
            if (ti < 0) continue;
            sum += snake(a.x[(size_t)ti * a.channels + c], al) * hf(a.w[c * a.kernel + k]);
        }
    }
    a.y[t] = tanhf(sum);
}

// The head for the decoder's 32 output channels, tiled over 32 * NO output rows:
// snake(x) of the rows and the left halo staged once in LDS, every load issued before
// the first is used. Eight lanes of four channels each compute NO consecutive
// outputs from NO + 6 rows (a 16-byte read a row for 28 products an output) and meet
// by DPP. (One thread per output, reading every channel and tap from LDS, was bound
// by those reads: 63.2 us at 483840 samples.)
template <int NO>
__global__ __launch_bounds__(256) void k_vae_head32_fm(VaeHeadArgs a) {
    constexpr uint32_t TB = 32u * NO, NR = TB + 6u, NS = (NR * 8u + 255u) / 256u;
    __shared__ __align__(16) float xs[NR * 32u];
    const uint32_t tid = threadIdx.x, g = tid & 7u, t0 = blockIdx.x * TB;
    float4 xv[NS];
#pragma unroll
    for (uint32_t i = 0; i < NS; ++i) {
        const uint32_t r = (tid >> 3) + 32u * i;
        const int t = (int)(t0 + r) - 6;
        xv[i] = r < NR && t >= 0 && (uint32_t)t < a.length
                    ? *reinterpret_cast<const float4 *>(a.x + (size_t)t * 32u + 4u * g)
                    : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float al[4], inv[4], w[7][4], big = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        al[e] = hf(a.alpha[4u * g + e]);
        inv[e] = snake_inv(al[e]);
#pragma unroll
        for (int k = 0; k < 7; ++k) w[k][e] = hf(a.w[(4u * g + e) * 7u + k]);
    }
#pragma unroll
    for (uint32_t i = 0; i < NS; ++i) {
        const uint32_t r = (tid >> 3) + 32u * i;
        const float v[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float s = al[e] * v[e];
            big = fmaxf(big, fabsf(s));
            o[e] = snake_fm(v[e], s, inv[e]);   // snake(0) = 0: the padding stays zero
        }
        if (r < NR) *reinterpret_cast<float4 *>(xs + r * 32u + 4u * g) = make_float4(o[0], o[1], o[2], o[3]);
    }
    if (any_large(big)) {
#pragma unroll 1
        for (uint32_t i = 0; i < 4u * NS; ++i) {
            const uint32_t r = (tid >> 3) + 32u * (i >> 2), c = 4u * g + (i & 3u);
            const int t = (int)(t0 + r) - 6;
            if (r >= NR || t < 0 || (uint32_t)t >= a.length) continue;
            const float v = a.x[(size_t)t * 32u + c], av = hf(a.alpha[c]);
            xs[r * 32u + c] = snake_any(v, av * v, snake_inv(av));
        }
    }
    __syncthreads();
    const uint32_t o0 = (tid >> 3) * NO;
    float acc[NO] = {};
#pragma unroll
    for (int r = 0; r < NO + 6; ++r) {
        const float4 q = *reinterpret_cast<const float4 *>(xs + (o0 + r) * 32u + 4u * g);
#pragma unroll
        for (int o = 0; o < NO; ++o) {
            const int k = r - o;
            if (k < 0 || k > 6) continue;
            acc[o] = fmaf(q.x, w[k][0], acc[o]);
            acc[o] = fmaf(q.y, w[k][1], acc[o]);
            acc[o] = fmaf(q.z, w[k][2], acc[o]);
            acc[o] = fmaf(q.w, w[k][3], acc[o]);
        }
    }
    float mine = 0.f;
#pragma unroll
    for (int o = 0; o < NO; ++o) {
        const float v = sum8(acc[o]);
        mine = g == (uint32_t)o ? v : mine;
    }
    const uint32_t t = t0 + o0 + g;
    if (g < (uint32_t)NO && t < a.length) a.y[t] = tanhf(mine + hf(a.b[0]));
}

// Other channel counts up to 48: one thread an output row, snake(x) of 256 rows and
// the left halo staged in LDS (row stride C + 1) with the conv weights.
__global__ __launch_bounds__(256) void k_vae_head_tiled_fm(VaeHeadArgs a) {
    __shared__ float xs[(256 + 6) * 49];
    __shared__ float ws[48 * 7];
    const uint32_t C = a.channels, S = C + 1u, t0 = blockIdx.x * 256u, halo = a.left_pad;
    const uint32_t n_st = (256u + halo) * C, tid = threadIdx.x;
    for (uint32_t i = tid; i < C * a.kernel; i += 256u) ws[i] = hf(a.w[i]);
    for (uint32_t idx = tid; idx < n_st; idx += 256u) {
        const uint32_t r = idx / C, c = idx - r * C;
        const int ti = (int)(t0 + r) - (int)halo;
        xs[r * S + c] = ti >= 0 && (uint32_t)ti < a.length ? snake(a.x[(size_t)ti * C + c], hf(a.alpha[c])) : 0.f;
    }
    __syncthreads();
    const uint32_t t = t0 + tid;
    if (t >= a.length) return;
    float sum = hf(a.b[0]);
    for (uint32_t c = 0; c < C; ++c)
        for (uint32_t k = 0; k < a.kernel; ++k) sum += xs[(tid + k) * S + c] * ws[c * a.kernel + k];
    a.y[t] = tanhf(sum);
}

unsigned grid1(uint64_t n) { return (unsigned)((n + 255u) / 256u); }

}  // namespace

int launch_vae_conv1d_cm(hipStream_t s, const VaeConvArgs &a, bool transpose) {
    if (!a.out_length || !a.out_channels) return VX_OK;
    const dim3 g(grid1(a.out_length), a.out_channels);
    if (transpose) {
        k_vae_convt1d_cm<<<g, 256, 0, s>>>(a);
        VX_LAUNCHED("k_vae_convt1d_cm");
    } else {
        k_vae_conv1d_cm<<<g, 256, 0, s>>>(a);
        VX_LAUNCHED("k_vae_conv1d_cm");
    }
    return VX_OK;
}

int launch_vae_snake_cm(hipStream_t s, const float *x, float *y, const void *alpha, uint32_t dtype, uint32_t c,
                        uint32_t len) {
    if (!c || !len) return VX_OK;
    k_vae_snake_cm<<<dim3(grid1(len), c), 256, 0, s>>>(x, y, alpha, dtype, c, len);
    VX_LAUNCHED("k_vae_snake_cm");
    return VX_OK;
}

int launch_vae_scale_bias_cm(hipStream_t s, float *x, const void *scale, const void *bias, uint32_t sdt,
                             uint32_t bdt, uint32_t c, uint32_t len, uint32_t bucket) {
    if (!c || !len) return VX_OK;
    k_vae_scale_bias_cm<<<dim3(grid1(len), c), 256, 0, s>>>(x, scale, bias, sdt, bdt, c, len, bucket);
    VX_LAUNCHED("k_vae_scale_bias_cm");
    return VX_OK;
}

int launch_vae_add_cm(hipStream_t s, float *a, const float *b, uint32_t c, uint32_t len) {
    if (!c || !len) return VX_OK;
    k_vae_add_cm<<<dim3(grid1(len), c), 256, 0, s>>>(a, b, c, len);
    VX_LAUNCHED("k_vae_add_cm");
    return VX_OK;
}

int launch_vae_tanh(hipStream_t s, float *x, uint32_t n) {
    if (!n) return VX_OK;
    k_vae_tanh<<<grid1(n), 256, 0, s>>>(x, n);
    VX_LAUNCHED("k_vae_tanh");
    return VX_OK;
}

int launch_vae_dwconv_fm(hipStream_t s, const VaeDwArgs &a) {
    const uint64_t n = (uint64_t)a.length * a.channels;
    if (!n) return VX_OK;
    if (a.yh && (!a.yl || a.channels % 32u)) return fail(VX_ERR_INVALID_ARG, "vae depthwise: planes need channels %% 32");
    if (a.kernel == 7u && a.left_pad == 6u * a.dilation && a.channels % 2u == 0u && n <= 1572864u &&
        ((uintptr_t)a.x & 7u) == 0 && ((uintptr_t)a.y & 7u) == 0) {
        k_vae_dw7_fm<<<grid1(n / 2u), 256, 0, s>>>(a);
        VX_LAUNCHED("k_vae_dw7_fm");
        return VX_OK;
    }
    if (a.kernel >= 1u && a.kernel <= 8u && a.left_pad == (a.kernel - 1u) * a.dilation && a.left_pad <= 54u) {
        const uint32_t CB = a.channels < 64u ? a.channels : 64u;   // >= 1; 2048 / CB rows per workgroup
        if ((CB & (CB - 1u)) == 0) {
            const uint32_t sh = (uint32_t)__builtin_ctz(CB), cblocks = (a.channels + CB - 1u) / CB;
            const uint32_t tb = 2048u >> sh;
            k_vae_dwconv_tiled_fm<8><<<dim3((a.length + tb - 1u) / tb, cblocks), 256, 0, s>>>(a, sh);
            VX_LAUNCHED("k_vae_dwconv_tiled_fm");
            return VX_OK;
        }
    }
    if (a.yh) return fail(VX_ERR_UNSUPPORTED, "vae depthwise: planes of this shape");
    k_vae_dwconv_fm<<<grid1(n), 256, 0, s>>>(a);
    VX_LAUNCHED("k_vae_dwconv_fm");
    return VX_OK;
}

int launch_vae_pre_fm(hipStream_t s, const float *x, float *y, const float *pre, uint32_t channels, uint32_t length) {
    const uint64_t n = (uint64_t)length * channels;
    if (!n) return VX_OK;
    if (channels % 4u == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15u) == 0)
        k_vae_pre_fm<4><<<grid1(n / 4u), 256, 0, s>>>(x, y, pre, channels, n);
    else
        k_vae_pre_fm<1><<<grid1(n), 256, 0, s>>>(x, y, pre, channels, n);
    VX_LAUNCHED("k_vae_pre_fm");
    return VX_OK;
}

int launch_vae_pre_planes(hipStream_t s, const float *x, const VaePlanes &y, const float *pre, uint32_t channels,
                          uint32_t length) {
    const uint64_t n = (uint64_t)length * channels;
    if (!n) return VX_OK;
    if (channels % 32u || !y.h || !y.l || y.block % 64u || y.block / 64u <= length ||
        ((uintptr_t)x | (uintptr_t)y.h | (uintptr_t)y.l | (uintptr_t)pre) & 15u || length > 0x3fffffffu)
        return fail(VX_ERR_INVALID_ARG, "vae pre: planes of %u channels, block %u", channels, y.block);
    k_vae_pre_planes<<<dim3(grid1(4ull * length), channels / 32u), 256, 0, s>>>(x, y, pre, channels, length);
    VX_LAUNCHED("k_vae_pre_planes");
    return VX_OK;
}

int launch_vae_repack_pre(hipStream_t s, const __half *scale, const __half *bias, const __half *alpha,
                          uint32_t channels, float *pre) {
    k_vae_repack_pre<<<grid1(channels), 256, 0, s>>>(scale, bias, alpha, channels, pre);
    VX_LAUNCHED("k_vae_repack_pre");
    return VX_OK;
}

int launch_vae_repack_convt(hipStream_t s, const __half *w, const __half *b, uint32_t cin, uint32_t cout,
                            uint32_t stride, uint32_t prefill_layout, __half *wp, float *bp) {
    const uint64_t rows = prefill_layout ? (stride * cout + 127u) / 128u * 128u : stride * cout;
    k_vae_repack_convt<<<grid1(rows * 2u * cin), 256, 0, s>>>(w, b, cin, cout, stride, prefill_layout, wp, bp);
    VX_LAUNCHED("k_vae_repack_convt");
    return VX_OK;
}

int launch_vae_linear_fm(hipStream_t s, const VaeLinearArgs &a) {
    if (!a.T || !a.N) return VX_OK;
    if (a.K > kVaeLinearMaxK) return fail(VX_ERR_UNSUPPORTED, "vae linear: K %u > %u", a.K, kVaeLinearMaxK);
    const bool chunks = a.K % 8u == 0 && (reinterpret_cast<uintptr_t>(a.w) & 15u) == 0;
    const uint32_t NB = a.N < 256u ? a.N : 256u, G = 256u / NB;
    uint32_t rpt = 8192u / (G * a.K);
    rpt = rpt < 1u ? 1u : (rpt > kLinRows ? kLinRows : rpt);
    const uint32_t RB = G * rpt;   // RB * K <= max(8192, G * K) floats
    if ((uint64_t)RB * a.K * 4u > 65536u)
        return fail(VX_ERR_UNSUPPORTED, "vae linear: %u rows x K %u exceed the LDS tile", RB, a.K);
    const dim3 grid((a.N + NB - 1u) / NB, (a.T + RB - 1u) / RB);
    if (chunks) {
        k_vae_linear_fm<<<grid, 256, (size_t)RB * a.K * 4u, s>>>(a, NB, RB);
        VX_LAUNCHED("k_vae_linear_fm");
    } else {
        k_vae_linear_fm_any<<<grid, 256, (size_t)RB * a.K * 4u, s>>>(a, NB, RB);
        VX_LAUNCHED("k_vae_linear_fm_any");
    }
    return VX_OK;
}

int launch_vae_head_fm(hipStream_t s, const VaeHeadArgs &a) {
    if (!a.length) return VX_OK;
    if (a.channels == 32u && a.left_pad == 6u && a.kernel == 7u && (reinterpret_cast<uintptr_t>(a.x) & 15u) == 0) {
        // 256 rows a workgroup once that gives every CU one, else 64.
        if (a.length >= 256u * 256u)
            k_vae_head32_fm<8><<<(a.length + 255u) / 256u, 256, 0, s>>>(a);
        else
            k_vae_head32_fm<2><<<(a.length + 63u) / 64u, 256, 0, s>>>(a);
        VX_LAUNCHED("k_vae_head32_fm");
        return VX_OK;
    }
    if (a.channels <= 48u && a.left_pad <= 6u && a.kernel == a.left_pad + 1u) {
        k_vae_head_tiled_fm<<<grid1(a.length), 256, 0, s>>>(a);
        VX_LAUNCHED("k_vae_head_tiled_fm");
        return VX_OK;
    }
    k_vae_head_fm<<<grid1(a.length), 256, 0, s>>>(a);
    VX_LAUNCHED("k_vae_head_fm");
    return VX_OK;
}

}  // namespace vx
