// AudioVAE residual unit of a decoder stage in one pass:
//   y[t][n] = x[t][n] + pb[n] + sum_c W[n][c] h[t][c]
//   h[t][c] = snake_a2(db[c] + sum_k dw[k][c] snake_a1(x[t + k d - 6 d][c])),  k < 7
// (audiovae.rs:400-407: snake, causal depthwise conv of dilation d, snake, 1x1 conv).
// The last unit of a stage also applies what the next transposed convolution does to
// its input, snake_pa(y * ps + pt), so that no pass of its own is needed for it.
//
// A workgroup covers TB rows and all C channels. For each block of KB channels it
// stages snake_a1(x) of its rows and their 6 d rows of history in LDS, writes h as
// f16 hi and lo planes into a second LDS tile and multiplies them with W
// (v_mfma_f32_32x32x16_f16, two products per step, f32 accumulation over the
// channel blocks). W is read in fragment order, 1 KB of consecutive bytes a load.
// The planes are kept [row][KB] with the 16-byte chunks of a row permuted by the row
// index, so that the A reads of 8 consecutive rows cover all banks.
//
// A pair of planes holds 22 bits of |h| < 65504 down to 2^-3, and 2^-25 absolutely below.
// Units of 32 and 64 channels, where f32 products are a choice, scale each row by a power
// of two into the planes and back after the products, so that neither the range nor
// small rows lose (22 bits of what is within 2^-18 of its row's largest). Cost: 3 us a
// unit at 252 frames (64 channels 41.0 -> 44.2, 32 channels 32.8 -> 35.5). Error of a
// decode against 64 bits, f32 products -> this: 1.7e-6 -> 1.5e-6, with h around 1e5 in
// these units 4.1e-6 -> 3.5e-6, around 1e-5 2.8e-6 -> 2.5e-6 (unscaled: not finite,
// 9e-3). Wider units keep the plain range of the GEMMs around them.
//
// Bound: x in and y out (8 bytes an element, 24 us a unit at 252 frames) against the
// two snakes' vector work (about 60 instructions an element with the history rows, as
// long again). Mean of the three units of a stage at 252 frames on MI355X, against a
// depthwise pass and a GEMM with atomic adds (256, 128 channels) or f32 products from
// LDS in one pass (64, 32): 256 channels 152 -> 63 us, 128 channels 110 -> 56, 64
// channels 91 -> 44, 32 channels 62 -> 35. Larger tiles of 256 and 128 channels at one
// workgroup of eight waves per CU were slower (79 and 60 us), and so was holding them
// to 128 vector registers for two (140 and 100 us: spills). The unit that ends a stage
// writes the next stage's planes: 12 us more at 256 channels (20 with an address a
// store), where a pass of its own over f32 would read and write 120 MB.
#include "vae_dev.h"

namespace vx {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float acc16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kMaxHalo = 54u;   // 6 * dilation 9

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

__device__ __forceinline__ float max4abs(float m, float4 v) {
    return fmaxf(fmaxf(fmaxf(m, fabsf(v.x)), fmaxf(fabsf(v.y), fabsf(v.z))), fabsf(v.w));
}
__device__ __forceinline__ float4 mul4(float4 a, float4 b) {
    return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
}
// x + sin(s)^2 * inv
__device__ __forceinline__ float4 snake4(float4 x, float4 s, float4 inv) {
    return make_float4(fmaf(sin_sq(s.x), inv.x, x.x), fmaf(sin_sq(s.y), inv.y, x.y), fmaf(sin_sq(s.z), inv.z, x.z),
                       fmaf(sin_sq(s.w), inv.w, x.w));
}

// A lane exchange inside a row of 16 lanes (gfx9 DPP controls).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}

// Offset (in halves) of channel c of a row in a plane of KB channels.
template <int KB>
__device__ __forceinline__ uint32_t plane_at(uint32_t row, uint32_t c) {
    const uint32_t sw = KB == 64 ? row & 7u : (row >> 1) & 3u;
    return row * KB + ((((c >> 3) ^ sw) << 3) | (c & 7u));
}

template <int C, int TB, int NW, int WM, int WN, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void k_vae_unit(VaeUnitArgs a) {
    constexpr int KB = C < 64 ? C : 64, NKB = C / KB, NT = 64 * NW;
    constexpr uint32_t G4 = KB / 4, RPP = NT / G4;              // float4 groups of a row, rows a pass
    constexpr int NS = (TB + kMaxHalo + RPP - 1) / RPP;         // staging passes
    constexpr int ND = (TB + RPP - 1) / RPP;                    // depthwise passes
    constexpr int MT = TB / 32 / WM, NTL = C / 32 / WN, KS = KB / 16;
    static_assert(MT * WM * 32 == TB && NTL * WN * 32 == C && WM * WN <= NW, "wave grid");
    __shared__ __attribute__((aligned(16))) float xs[(TB + kMaxHalo) * KB];
    __shared__ __attribute__((aligned(16))) _Float16 ph[TB * KB];
    __shared__ __attribute__((aligned(16))) _Float16 pl[TB * KB];
    // Up to 64 channels a block is the whole row: the row's largest |h| is brought into
    // [2^14, 2^15), and un[row] takes that back.
    constexpr bool kScaled = NKB == 1;
    __shared__ __attribute__((aligned(16))) float un[kScaled ? TB : 4];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, l32 = lane & 31u, hs = lane >> 5;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wv / WN, wn = wv % WN;
    const bool mul = wv < (uint32_t)(WM * WN);
    if (a.pre && blockIdx.x == 0) {   // row -1 of the planes
        for (uint32_t i = tid; i < (uint32_t)C / 4u; i += NT) {   // plane, block, 16-byte chunk
            __half *const p = (i & 4u ? a.planes.l : a.planes.h) + (size_t)(i >> 3) * (a.planes.block / 2u);
            *reinterpret_cast<uint4 *>(p - 32 + 8 * (int)(i & 3u)) = make_uint4(0, 0, 0, 0);
        }
    }
    const uint32_t t0 = blockIdx.x * TB, halo = 6u * a.dilation, rows = TB + halo;
    const uint32_t c4 = 4u * (tid % G4), r0 = tid / G4;
    // Uniform bases with 32-bit offsets: rows of the tile from its history on (rows
    // before 0 are not read), and from its first row on.
    const float *const xh = a.x + ((int64_t)t0 - (int64_t)halo) * C, *const xt = a.x + (size_t)t0 * C;
    float *const yt = a.y + (size_t)t0 * C;
    const uint32_t skip = t0 < halo ? halo - t0 : 0u;                             // first staged row >= 0
    const uint32_t have = a.length - t0 < (uint32_t)TB ? a.length - t0 : TB;      // rows of the tile
    const uint32_t end = have + halo;
    const bool full = skip == 0 && have == (uint32_t)TB;   // the common tile: no row to leave out

    acc16 acc[MT][NTL] = {};
#pragma unroll 1
    for (uint32_t kb = 0; kb < (uint32_t)NKB; ++kb) {
        // Uniform bases of this block, opaque so that the loads keep them in scalar
        // registers with one lane offset instead of an address each in vector ones.
        const float *pk = a.p + kb * (kVaeUnitParams * KB);
        const __half *wk0 = a.w + ((size_t)(wn * NTL) * (C / 16) + kb * KS) * 512u;
        asm volatile("" : "+s"(pk), "+s"(wk0));
        float4 xv[NS];
        const float *xk = xh + kb * KB;
        if (full) {
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                uint32_t r = r0 + RPP * i;
                if ((i + 1) * (int)RPP > TB) r = r < rows ? r : rows - 1u;   // loaded, not used
                xv[i] = ld4(xk + (r * C + c4));
            }
        } else {
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                const uint32_t r = r0 + RPP * i;
                xv[i] = r >= skip && r < end ? ld4(xk + (r * C + c4)) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
        {
            const float4 a1 = ld4(pk + c4), i1 = ld4(pk + KB + c4);
            float big = 0.f;
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                const uint32_t r = r0 + RPP * i;
                if (r < rows) {
                    const float4 s = mul4(a1, xv[i]);
                    big = max4abs(big, s);
                    *reinterpret_cast<float4 *>(xs + r * KB + c4) = snake4(xv[i], s, i1);   // snake(0) = 0
                }
            }
            if (any_large(big)) {
#pragma unroll 1
                for (uint32_t i = 4u * r0; i < 4u * end; i = (i & 3u) == 3u ? i - 3u + 4u * RPP : i + 1u) {
                    const uint32_t r = i >> 2, ce = c4 + (i & 3u);
                    if (r < skip) continue;
                    const float v = xh[kb * KB + (r * C + ce)];
                    xs[r * KB + ce] = fmaf(sin_sq_any(pk[ce] * v), pk[KB + ce], v);
                }
            }
        }
        __syncthreads();
        // The products' weights of this block, in flight during the depthwise taps.
        h8 wf[NTL][KS];
        if (mul) {
#pragma unroll
            for (int n = 0; n < NTL; ++n)
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    wf[n][k] = *reinterpret_cast<const h8 *>(wk0 + (n * (C / 16) + k) * 512 + lane * 8u);
        }
        {
            const float4 a2 = ld4(pk + 2 * KB + c4), i2 = ld4(pk + 3 * KB + c4), db = ld4(pk + 4 * KB + c4);
            float4 wk[7];
#pragma unroll
            for (int k = 0; k < 7; ++k) wk[k] = ld4(pk + (6 + k) * KB + c4);
            auto conv = [&](uint32_t r) {
                float4 s = db;
#pragma unroll
                for (int k = 0; k < 7; ++k) {
                    const float4 v = *reinterpret_cast<const float4 *>(xs + (r + k * a.dilation) * KB + c4);
                    s.x = fmaf(v.x, wk[k].x, s.x);
                    s.y = fmaf(v.y, wk[k].y, s.y);
                    s.z = fmaf(v.z, wk[k].z, s.z);
                    s.w = fmaf(v.w, wk[k].w, s.w);
                }
                return s;
            };
            auto put = [&](uint32_t r, float4 v) {
                if constexpr (kScaled) {
                    // The largest of the row's G4 lanes, as bits (they order like the values).
                    uint32_t m = max(__builtin_bit_cast(uint32_t, max4abs(0.f, v)), 15u << 23);
                    m = max(m, dpp_u<0xb1>(m));    // quad_perm [1,0,3,2]
                    m = max(m, dpp_u<0x4e>(m));    // quad_perm [2,3,0,1]
                    m = max(m, dpp_u<0x141>(m));   // row_half_mirror
                    if constexpr (G4 == 16) m = max(m, dpp_u<0x140>(m));   // row_mirror
                    m &= 0x7f800000u;   // 2^(14 - e), and 2^(e - 14) to come back, of exponent e >= -112
                    const float sc = __builtin_bit_cast(float, (268u << 23) - m);
                    v = make_float4(v.x * sc, v.y * sc, v.z * sc, v.w * sc);
                    if (tid % G4 == 0u) un[r] = __builtin_bit_cast(float, m - (14u << 23));
                }
                const h4 h = {(_Float16)v.x, (_Float16)v.y, (_Float16)v.z, (_Float16)v.w};
                const h4 l = {(_Float16)(v.x - (float)h[0]), (_Float16)(v.y - (float)h[1]),
                              (_Float16)(v.z - (float)h[2]), (_Float16)(v.w - (float)h[3])};
                const uint32_t o = plane_at<KB>(r, c4);
                *reinterpret_cast<h4 *>(ph + o) = h;
                *reinterpret_cast<h4 *>(pl + o) = l;
            };
            float big = 0.f;
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                const uint32_t r = r0 + RPP * i;
                if (TB % RPP == 0 || r < (uint32_t)TB) {
                    const float4 u = conv(r), s = mul4(a2, u);
                    big = max4abs(big, s);
                    put(r, snake4(u, s, i2));
                }
            }
            if (any_large(big)) {
                if constexpr (kScaled) {
#pragma unroll 1
                    for (uint32_t r = r0; r < (uint32_t)TB; r += RPP) {
                        const float4 u = conv(r);
                        float4 v = u, s = mul4(a2, u), q = i2;
#pragma unroll 1
                        for (int j = 0; j < 4; ++j) {   // the four channels in turn through the first place
                            const float h = fmaf(sin_sq_any(s.x), q.x, v.x);
                            v = make_float4(v.y, v.z, v.w, h);
                            s = make_float4(s.y, s.z, s.w, s.x);
                            q = make_float4(q.y, q.z, q.w, q.x);
                        }
                        put(r, v);
                    }
                } else {
#pragma unroll 1
                    for (uint32_t i = 4u * r0; i < 4u * TB; i = (i & 3u) == 3u ? i - 3u + 4u * RPP : i + 1u) {
                        const uint32_t r = i >> 2, ce = c4 + (i & 3u);
                        float u = pk[4 * KB + ce];
#pragma unroll 1
                        for (uint32_t k = 0; k < 7u; ++k)
                            u = fmaf(xs[(r + k * a.dilation) * KB + ce], pk[(6u + k) * KB + ce], u);
                        u = fmaf(sin_sq_any(pk[2 * KB + ce] * u), pk[3 * KB + ce], u);
                        const _Float16 h = (_Float16)u;
                        ph[plane_at<KB>(r, ce)] = h;
                        pl[plane_at<KB>(r, ce)] = (_Float16)(u - (float)h);
                    }
                }
            }
        }
        __syncthreads();
        if (mul) {
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    const uint32_t o = plane_at<KB>(32u * (wm * MT + m) + l32, 16u * k + 8u * hs);
                    const h8 xh = *reinterpret_cast<const h8 *>(ph + o), xl = *reinterpret_cast<const h8 *>(pl + o);
#pragma unroll
                    for (int n = 0; n < NTL; ++n) {
                        acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xh, wf[n][k], acc[m][n], 0, 0, 0);
                        acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xl, wf[n][k], acc[m][n], 0, 0, 0);
                    }
                }
        }
    }
    if (!mul) return;
    if constexpr (kScaled) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                const float4 f = ld4(un + 32 * (wm * MT + m) + 8 * (r >> 2) + 4 * hs);
#pragma unroll
                for (int n = 0; n < NTL; ++n) {
                    acc[m][n][r] *= f.x;
                    acc[m][n][r + 1] *= f.y;
                    acc[m][n][r + 2] *= f.z;
                    acc[m][n][r + 3] *= f.w;
                }
            }
    }

    // Lane (l32, hs) holds channel n = 32 tile + l32 of rows 8 (r / 4) + 4 hs + r % 4.
    const uint32_t tb = 32u * wm * MT + 4u * hs;
    auto each = [&](auto f) {   // f(channel tile, row, offset from the tile's first value, value) -> new value
#pragma unroll
        for (int n = 0; n < NTL; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t t = tb + 32u * m + 8u * (r >> 2) + (r & 3);
                    acc[m][n][r] = f(n, t, t * C + 32u * (wn * NTL + n) + l32, acc[m][n][r]);
                }
    };
    float pb[NTL], ws[NTL];
#pragma unroll
    for (int n = 0; n < NTL; ++n) {
        const uint32_t ch = 32u * (wn * NTL + n) + l32;
        const float *const q = a.p + ch / KB * (kVaeUnitParams * KB) + ch % KB;
        pb[n] = q[5 * KB], ws[n] = q[13 * KB];
    }
    if (full)
        each([&](int n, uint32_t, uint32_t o, float v) { return xt[o] + fmaf(v, ws[n], pb[n]); });
    else
        each([&](int n, uint32_t t, uint32_t o, float v) { return (t < have ? xt[o] : 0.f) + fmaf(v, ws[n], pb[n]); });
    auto store = [&]() {
        if (full)
            each([&](int, uint32_t, uint32_t o, float v) { return yt[o] = v; });
        else
            each([&](int, uint32_t t, uint32_t o, float v) {
                if (t < have) yt[o] = v;
                return v;
            });
    };
    if (!a.pre) {
        store();
        return;
    }
    // The next stage's planes. A row's 32 channels are one 64-byte run per plane, its
    // 16-byte chunks permuted by the row; lanes pair up, the even one storing both high
    // halves and the odd one both low halves.
    const VaePlanes &P = a.planes;
    auto po = [&](int n, uint32_t t) {   // halves from the tile's row 0 of block 0, this lane's channel
        return (size_t)(wn * NTL + n) * (P.block / 2u) + t * 32u +
               8u * ((l32 >> 3) ^ xperm(t)) + (l32 & 7u);
    };
    __half *const yh = P.h + (size_t)t0 * 32u, *const yl = P.l + (size_t)t0 * 32u;
    float ps[NTL], pt[NTL], pa[NTL], pi[NTL], big = 0.f;
#pragma unroll
    for (int n = 0; n < NTL; ++n) {
        const uint32_t ch = 32u * (wn * NTL + n) + l32;
        ps[n] = a.pre[ch], pt[n] = a.pre[C + ch], pa[n] = a.pre[2 * C + ch], pi[n] = a.pre[3 * C + ch];
    }
    each([&](int n, uint32_t, uint32_t, float v) {
        v = fmaf(v, ps[n], pt[n]);
        big = fmaxf(big, fabsf(pa[n] * v));
        return v;
    });
    if (any_large(big)) {
        // The bits are stored unfinished (upper half in one plane, lower in the other),
        // then finished one by one by the same lane.
        each([&](int n, uint32_t t, uint32_t, float v) {
            if (t < have) {
                const uint32_t b = __builtin_bit_cast(uint32_t, v);
                yh[po(n, t)] = __builtin_bit_cast(__half, (unsigned short)(b >> 16));
                yl[po(n, t)] = __builtin_bit_cast(__half, (unsigned short)b);
            }
            return v;
        });
#pragma unroll 1
        for (uint32_t i = 0; i < (uint32_t)(NTL * MT * 16); ++i) {
            const uint32_t n = i / (MT * 16), m = i / 16 % MT, r = i % 16;
            const uint32_t ch = 32u * (wn * NTL + n) + l32, t = tb + 32u * m + 8u * (r >> 2) + (r & 3);
            if (t >= have) continue;
            const size_t o = po((int)n, t);
            float v = __builtin_bit_cast(float, (uint32_t)__builtin_bit_cast(unsigned short, yh[o]) << 16 |
                                                    __builtin_bit_cast(unsigned short, yl[o]));
            v = fmaf(sin_sq_any(a.pre[2 * C + ch] * v), a.pre[3 * C + ch], v);
            const _Float16 h = (_Float16)v;
            yh[o] = __builtin_bit_cast(__half, h);
            yl[o] = __builtin_bit_cast(__half, (_Float16)(v - (float)h));
        }
        return;
    }
    const uint32_t odd = lane & 1u, sel = odd ? 0x03020706u : 0x05040100u;   // of (other, own)
    // Row 4 hs + 8 q + j of 32 has chunk (l32 / 8) ^ 2 hs ^ (q ^ j / 2): four lane
    // addresses a channel tile, and the rows are immediate offsets from them.
    __half *yx[NTL][4];
#pragma unroll
    for (int n = 0; n < NTL; ++n)
#pragma unroll
        for (uint32_t x = 0; x < 4u; ++x)
            yx[n][x] = (odd ? yl : yh) - odd + (size_t)(wn * NTL + n) * (P.block / 2u) + tb * 32u +
                       8u * ((l32 >> 3) ^ (2u * hs) ^ x) + (l32 & 7u);
    auto finish = [&](auto keep) {
#pragma unroll
        for (int n = 0; n < NTL; ++n)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = 32 * m + 8 * (r >> 2) + (r & 3);
                    const float v = fmaf(sin_sq(pa[n] * acc[m][n][r]), pi[n], acc[m][n][r]);
                    const _Float16 h = (_Float16)v, l = (_Float16)(v - (float)h);
                    const uint32_t own = (uint32_t)__builtin_bit_cast(unsigned short, h) |
                                         (uint32_t)__builtin_bit_cast(unsigned short, l) << 16;
                    const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)own, 0xB1, 0xf, 0xf, true);
                    if (keep(tb + row))
                        *reinterpret_cast<uint32_t *>(yx[n][(r >> 2) ^ ((r & 3) >> 1)] + 32 * row) =
                            __builtin_amdgcn_perm(other, own, sel);
                }
    };
    if (full)
        finish([](uint32_t) { return true; });
    else
        finish([&](uint32_t t) { return t < have; });
}

// A unit's parameters as f32 [C / KB][14][KB], KB = min(C, 64): a1, 1/(a1 + 1e-9), a2,
// 1/(a2 + 1e-9), db, pb, dw[7], ws; and its 1x1 weight in fragment order: block (n / 32,
// c / 16) of 64 lanes x 8 halves, lane l holding row n % 32 = l % 32, columns 8 (l / 32)...
// Rows of the weight are multiplied by the power of two 1/ws that brings their largest
// value into [2^14, 2^15): exact, and no weight is left subnormal whose products the
// matrix cores would sum with fewer bits (error of a decode with weights of 2e-6 against
// 64 bits: 8.0e-6 as they are, 3.5e-6 so, 4.1e-6 with f32 products). One workgroup a row.
__global__ __launch_bounds__(256) void k_vae_repack_unit(const __half *a1, const __half *dw, const __half *db,
                                                         const __half *a2, const __half *pw, const __half *pb,
                                                         uint32_t C, float *p, __half *w) {
    __shared__ float part[4];
    const uint32_t n = blockIdx.x, tid = threadIdx.x, KB = C < 64u ? C : 64u;
    const __half *const row = pw + (size_t)n * C;
    float m = 0.f;
    for (uint32_t c = tid; c < C; c += 256u) m = fmaxf(m, fabsf(vae_h2f(row[c])));
#pragma unroll
    for (int d = 32; d; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
    if ((tid & 63u) == 0u) part[tid >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
    int k = 0;   // 2^k m in [2^14, 2^15)
    if (m > 0.f && m < 32768.0f) k = 14 - (int)((__builtin_bit_cast(uint32_t, m) >> 23) - 127u);
    const float up = __builtin_bit_cast(float, (uint32_t)(127 + k) << 23);
    for (uint32_t c = tid; c < C; c += 256u) {
        const uint32_t l = (n & 31u) + 32u * ((c >> 3) & 1u), b = n / 32u * (C / 16u) + c / 16u;
        w[b * 512u + l * 8u + (c & 7u)] = __builtin_bit_cast(__half, (_Float16)(up * vae_h2f(row[c])));
    }
    if (tid) return;
    float *const q = p + n / KB * (kVaeUnitParams * KB) + n % KB;
    q[0] = vae_h2f(a1[n]);
    q[KB] = snake_inv(vae_h2f(a1[n]));
    q[2u * KB] = vae_h2f(a2[n]);
    q[3u * KB] = snake_inv(vae_h2f(a2[n]));
    q[4u * KB] = vae_h2f(db[n]);
    q[5u * KB] = vae_h2f(pb[n]);
    for (uint32_t i = 0; i < 7u; ++i) q[(6u + i) * KB] = vae_h2f(dw[n * 7u + i]);
    q[13u * KB] = __builtin_bit_cast(float, (uint32_t)(127 - k) << 23);
}

template <int C, int TB, int NW, int WM, int WN, int OCC>
int launch_unit(hipStream_t s, const VaeUnitArgs &a) {
    k_vae_unit<C, TB, NW, WM, WN, OCC><<<(a.length + TB - 1u) / TB, 64 * NW, 0, s>>>(a);
    VX_LAUNCHED("k_vae_unit");
    return VX_OK;
}

}  // namespace

bool vae_unit_channels(uint32_t c) { return c == 32u || c == 64u || c == 128u || c == 256u || c == 512u; }

int launch_vae_repack_unit(hipStream_t s, const __half *a1, const __half *dw, const __half *db, const __half *a2,
                           const __half *pw, const __half *pb, uint32_t channels, float *p, __half *w) {
    k_vae_repack_unit<<<channels, 256, 0, s>>>(a1, dw, db, a2, pw, pb, channels, p, w);
    VX_LAUNCHED("k_vae_repack_unit");
    return VX_OK;
}

int launch_vae_unit(hipStream_t s, const VaeUnitArgs &a) {
    if (!a.length) return VX_OK;
    if (!vae_unit_channels(a.channels) || !a.dilation || 6u * a.dilation > kMaxHalo || a.x == a.y)
        return fail(VX_ERR_UNSUPPORTED, "vae residual unit: %u channels, dilation %u", a.channels, a.dilation);
    if (a.pre && (!a.planes.h || !a.planes.l || a.planes.block % 64u || a.planes.block / 64u <= a.length))
        return fail(VX_ERR_INVALID_ARG, "vae residual unit: planes of %u rows, block %u", a.length, a.planes.block);
    // Tiles of 128 or 64 rows (less history per row) once they give every CU one, else
    // of 32 (4 frames, 256 channels: 15 workgroups of 64 rows on 256 CUs).
    switch (a.channels) {
    case 32:
        return a.length >= 128u * 256u ? launch_unit<32, 128, 4, 4, 1, 4>(s, a) : launch_unit<32, 32, 4, 1, 1, 2>(s, a);
    case 64:
        return a.length >= 128u * 256u ? launch_unit<64, 128, 8, 4, 2, 4>(s, a) : launch_unit<64, 32, 4, 1, 2, 2>(s, a);
    case 128:
        return a.length >= 64u * 256u ? launch_unit<128, 64, 4, 1, 4, 2>(s, a) : launch_unit<128, 32, 4, 1, 4, 2>(s, a);
    case 512:
        return launch_unit<512, 32, 8, 1, 8, 2>(s, a);
    default:
        return a.length >= 64u * 256u ? launch_unit<256, 64, 4, 1, 4, 2>(s, a) : launch_unit<256, 32, 8, 1, 8, 2>(s, a);
    }
}

}  // namespace vx
