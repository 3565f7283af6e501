// Projections of a short prefill chunk on gfx950 (T <= 128 rows, usually a prompt of
// a few words or the last chunk of a long one): Q8_0 or F16 weights in the prefill
// layout, X as tiled hi/lo planes, the arithmetic of k_gemm_pf (kernels_gemm.hip):
//   C[t][n] = sum_b d[n][b] * sum_{k in b} q * (x_hi + x_lo)
//
// At so few rows a launch is bound by how fast a CU takes operands in: the weights once
// (25 MB of Q8_0 for gate/up at the VoxCPM2 geometry, 5 us at the copy rate) and X, from
// the L2, by every workgroup. So the work is split for bytes in flight:
//   * a workgroup owns 32 weight rows (two 16-row fragments), or 32 gate rows and their
//     up rows, and every token; its waves take interleaved 32-column blocks of its K
//     range, and each keeps DEPTH blocks of operands in flight in registers;
//   * both stored layouts are read as they are: 16 rows of one 32-column block are 512
//     contiguous bytes of quants (1 KB of f16), permuted only inside, which is one
//     operand of v_mfma_f32_16x16x32_f16 with the lane's chunk picked by the
//     permutation. A Q8_0 block is one MFMA step, so its products start from zero and
//     enter the sums scaled by the block's f32 scale;
//   * the partial tiles of the waves meet in LDS; split K leaves slabs that the consumer
//     sums.
// Against k_gemm (64-token tiles, at most four splits, atomic sums) four Q8_0 layers
// took on MI355X at 2 / 16 / 37 / 64 / 127 rows 381 / 409 / 431 / 435 / 448 ->
// 193 / 207 / 268 / 308 / 429 us, F16 381 / 406 / 431 / 434 / 448 -> 206 / 221 / 281 /
// 318 / 427; with the RoPE and norm kernels of today 180 / 197 / 258 / 298 / 412 and
// 195 / 212 / 273 / 311 / 416. Gate/up at 37 rows: 17 us with 64 rows a workgroup, 22
// with 32 (every workgroup reads all of X), 26 with 128 (too few workgroups); eight
// waves: 18. The split projections are the other way round (their K ranges are short):
// 9 us with 32 rows, 11 with 64; one workgroup per CU beat two (X again) by 10%.
#include "quant_dev.h"
#include "vae_dev.h"

namespace vx {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int NW = 4;             // waves per workgroup
constexpr uint32_t kPiece = 128;  // weight rows and tokens of a stored tile

__device__ __forceinline__ h8 widen(u2v u) {
    const uint2 lo = q8x4_to_f16(u[0]), hi = q8x4_to_f16(u[1]);
    return __builtin_bit_cast(h8, u4v{lo.x, lo.y, hi.x, hi.y});
}

__device__ __forceinline__ f4 mfma16(h8 a, h8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

template <int WK, int MT, int NF>
struct Ops {
    u4v xh[MT], xl[MT];
    u4v w[NF];
};
template <int MT, int NF>
struct Ops<WT_Q8, MT, NF> {
    u4v xh[MT], xl[MT];
    u2v w[NF];
    float d[NF];
};

// Grid: a.ntn row tiles x a.ntm token tiles x a.ksplit K ranges. XB: block-major planes.
template <int WK, int EPI, int MT, int NF, bool XB>
__global__ __launch_bounds__(64 * NW) void k_gemm_ps(GemmArgs a) {
    constexpr uint32_t kRows = 16u * NF;   // weight rows of the workgroup
    __shared__ f4 red[NW / 2][MT][NF][64];   // partial tiles [wave][token fragment][row fragment][lane]
    constexpr int DEPTH = MT <= 4 ? 4 : 3;
    const uint32_t tile = blockIdx.x % a.ntn, ks = blockIdx.x / a.ntn / a.ntm;
    const uint32_t m0 = blockIdx.x / a.ntn % a.ntm * (16u * MT);   // first token
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r16 = lane & 15u, g = lane >> 4;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t seg = 0;
    if constexpr (EPI != GEPI_SWIGLU) {
        while (seg + 1 < a.nseg && tile >= a.seg[seg + 1].tile0) ++seg;
    }
    const GemmSeg &sg = a.seg[seg];
    const uint32_t nblk = a.K >> 5;
    // A gate/up tile is stored as 32 gate rows (fragments 0 and 1) and their up rows; padding rows of the last tile are stored as zeros.
    const uint8_t *wr[NF];
    const float *dr[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        const uint32_t r0 = kRows * (tile - sg.tile0) + 16u * f;
        const uint32_t n = (r0 & (kPiece - 1u)) + r16;
        const size_t piece = (size_t)(r0 / kPiece) * nblk;
        const uint8_t *base = reinterpret_cast<const uint8_t *>(sg.pq);
        wr[f] = WK == WT_Q8 ? base + piece * (kPiece * 32u) + n * 32u + 8u * (g ^ wperm(n))
                            : base + piece * (kPiece * 64u) + n * 64u + 16u * (g ^ xperm(n));
        dr[f] = WK == WT_Q8 ? sg.pd + piece * kPiece + n : nullptr;
    }
    const uint8_t *const xh = reinterpret_cast<const uint8_t *>(a.xh), *const xl = reinterpret_cast<const uint8_t *>(a.xl);
    // Rows past T of the 128-row tile are multiplied and never stored. Rows read one
    // earlier (xs) carry the permutation of that row.
    uint32_t xo[MT], xs[XB ? MT : 1];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const uint32_t t = m0 + 16u * mt + r16;
        const uint32_t row = XB ? t * 64u : (t / kPiece * nblk * kPiece + t % kPiece) * 64u;
        xo[mt] = row + 16u * (g ^ xperm(t));
        if constexpr (XB) xs[mt] = row + 16u * (g ^ xperm(t - 1u));
    }
    const uint32_t s0 = ks * nblk / a.ksplit, s1 = (ks + 1u) * nblk / a.ksplit;
    const int n_it = s0 + wv < s1 ? (int)((s1 - s0 - wv + NW - 1u) / NW) : 0;

    f4 acc[MT][NF];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[mt][f] = f4{0.f, 0.f, 0.f, 0.f};
    Ops<WK, MT, NF> ring[DEPTH];
    auto load = [&](Ops<WK, MT, NF> &o, int i) {
        const size_t blk = s0 + wv + NW * (uint32_t)i;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if constexpr (WK == WT_Q8) {
                o.w[f] = __builtin_nontemporal_load(reinterpret_cast<const u2v *>(wr[f] + blk * (kPiece * 32u)));
                o.d[f] = __builtin_nontemporal_load(dr[f] + blk * kPiece);
            } else {
                o.w[f] = __builtin_nontemporal_load(reinterpret_cast<const u4v *>(wr[f] + blk * (kPiece * 64u)));
            }
        }
        const bool shifted = XB && blk < a.x_shift;
        const ptrdiff_t xb = !XB       ? (ptrdiff_t)(blk * (kPiece * 64u))
                             : shifted ? (ptrdiff_t)(blk * a.x_block) - 64
                                       : (ptrdiff_t)((blk - a.x_shift) * a.x_block);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const uint32_t x = XB && shifted ? xs[XB ? mt : 0] : xo[mt];
            o.xh[mt] = *reinterpret_cast<const u4v *>(xh + xb + x);
            o.xl[mt] = *reinterpret_cast<const u4v *>(xl + xb + x);
        }
    };
    auto mma = [&](const Ops<WK, MT, NF> &o) {
        h8 b[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            if constexpr (WK == WT_Q8)
                b[f] = widen(o.w[f]);
            else
                b[f] = __builtin_bit_cast(h8, o.w[f]);
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const h8 ah = __builtin_bit_cast(h8, o.xh[mt]), al = __builtin_bit_cast(h8, o.xl[mt]);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                if constexpr (WK == WT_Q8) {
                    const f4 p = mfma16(al, b[f], mfma16(ah, b[f], f4{0.f, 0.f, 0.f, 0.f}));
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[mt][f][r] = fmaf(o.d[f], p[r], acc[mt][f][r]);
                } else {
                    acc[mt][f] = mfma16(al, b[f], mfma16(ah, b[f], acc[mt][f]));
                }
            }
        }
    };
    // Loads are unconditional (past the wave's last block they repeat it): under a
    // branch the compiler would wait for everything in flight before each MFMA.
    if (n_it > 0) {
#pragma unroll
        for (int u = 0; u < DEPTH - 1; ++u) load(ring[u], min(u, n_it - 1));
        for (int it = 0; it < n_it; it += DEPTH) {
#pragma unroll
            for (int u = 0; u < DEPTH; ++u) {
                const int i = it + u;
                load(ring[(u + DEPTH - 1) % DEPTH], min(i + DEPTH - 1, n_it - 1));
                if (i < n_it) mma(ring[u]);
            }
        }
    }
    // Lane (r16, g) holds tokens 4g .. 4g + 3 of its token fragment for weight row r16.
    if (wv >= NW / 2) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < NF; ++f) red[wv - NW / 2][mt][f][lane] = acc[mt][f];
    }
    __syncthreads();
    if (wv < NW / 2) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < NF; ++f) red[wv][mt][f][lane] += acc[mt][f];
    }
    __syncthreads();
    auto part = [&](uint32_t tok, uint32_t f, uint32_t n) {
        const uint32_t ln = n + 16u * ((tok >> 2) & 3u), mt = tok >> 4, r = tok & 3u;
        float v = red[0][mt][f][ln][r];
#pragma unroll
        for (int w = 1; w < NW / 2; ++w) v += red[w][mt][f][ln][r];
        return v;
    };
    if constexpr (EPI == GEPI_SWIGLU) {
        constexpr uint32_t kPairs = kRows / 2u;
        for (uint32_t o = tid; o < kPairs * 16u * MT; o += 64u * NW) {
            const uint32_t nl = o % kPairs, tok = o / kPairs, row = kPairs * tile + nl, f = nl >> 4, n = nl & 15u;
            if (m0 + tok >= a.T || row >= sg.rows) continue;
            const float gv = part(tok, f, n), uv = part(tok, f + 2u, n);
            const float v = gv / (1.0f + expf(-gv)) * uv;   // matvec_swiglu.comp:67
            const size_t po = tiled_plane_index(m0 + tok, row, a.ldp);
            const _Float16 hv = (_Float16)v;
            a.oh[po] = __builtin_bit_cast(__half, hv);
            a.ol[po] = __builtin_bit_cast(__half, (_Float16)(v - (float)hv));
        }
    } else {
        const bool slab = a.ksplit > 1u;
        float *const out = EPI == GEPI_STORE ? sg.out + (slab ? ks * a.ws_stride : 0u)
                           : slab            ? a.ws + ks * a.ws_stride
                                             : sg.out;
        for (uint32_t o = tid; o < kRows * 16u * MT; o += 64u * NW) {
            const uint32_t nl = o % kRows, tok = o / kRows, row = kRows * (tile - sg.tile0) + nl;
            if (m0 + tok >= a.T || row >= sg.rows) continue;
            float v = part(tok, nl >> 4, nl & 15u);
            if constexpr (WK == WT_F16) {
                if (sg.bias && ks == 0u)
                    v += sg.bias_dtype == 0 ? static_cast<const float *>(sg.bias)[row]
                                            : __half2float(static_cast<const __half *>(sg.bias)[row]);
            }
            float *const dst = out + (size_t)(m0 + tok) * sg.ldo + row;
            if constexpr (EPI == GEPI_RESIDUAL && NF == 1) {
                if (a.pre) {
                    const float y = fmaf(*dst + v, a.pre[row], a.pre[sg.rows + row]), sn = a.pre[2u * sg.rows + row] * y;
                    const float sq = fabsf(sn) < kSinSqMax ? sin_sq(sn) : sin_sq_any(sn);
                    const float p = fmaf(sq, a.pre[3u * sg.rows + row], y);
                    const _Float16 hv = (_Float16)p;
                    const uint32_t t = m0 + tok;
                    const size_t po = (size_t)(row >> 5) * (a.o_block / 2u) + (size_t)t * 32u +
                                      8u * (((row >> 3) & 3u) ^ xperm(t)) + (row & 7u);
                    a.oh[po] = __builtin_bit_cast(__half, hv);
                    a.ol[po] = __builtin_bit_cast(__half, (_Float16)(p - (float)hv));
                    if (t == 0u) {
                        const ptrdiff_t z = (ptrdiff_t)((size_t)(row >> 5) * (a.o_block / 2u) + (row & 31u)) - 32;
                        a.oh[z] = a.ol[z] = __float2half(0.f);
                    }
                    continue;
                }
            }
            if constexpr (EPI == GEPI_STORE)
                *dst = v * a.alpha;
            else
                *dst = slab ? v * a.scale : *dst + v * a.scale;
        }
    }
}

#define VX_PS_CASE(M, NF, XB)                                                    \
    if (mt == M) {                                                               \
        k_gemm_ps<WK, EPI, M, NF, XB><<<grid, 64 * NW, 0, s>>>(a);               \
        VX_LAUNCHED("k_gemm_ps");                                                \
        return VX_OK;                                                            \
    }
// One token tile of up to 128 rows.
template <int WK, int EPI>
int launch_ps(hipStream_t s, const GemmArgs &a, uint32_t grid) {
    constexpr int NF = EPI == GEPI_SWIGLU ? 4 : 2;
    const uint32_t mt = (a.T + 15u) / 16u;
    VX_PS_CASE(1, NF, false)
    VX_PS_CASE(2, NF, false)
    VX_PS_CASE(3, NF, false)
    VX_PS_CASE(4, NF, false)
    VX_PS_CASE(5, NF, false)
    VX_PS_CASE(6, NF, false)
    VX_PS_CASE(7, NF, false)
    VX_PS_CASE(8, NF, false)
    return fail(VX_ERR_UNSUPPORTED, "short prefill gemm: %u rows", a.T);
}
// Token tiles of mt fragments.
template <int EPI, int NF, bool XB>
int launch_ps_tiles(hipStream_t s, const GemmArgs &a, uint32_t grid, uint32_t mt) {
    constexpr int WK = WT_F16;
    VX_PS_CASE(1, NF, XB)
    VX_PS_CASE(2, NF, XB)
    VX_PS_CASE(4, NF, XB)
    return fail(VX_ERR_UNSUPPORTED, "short gemm: token tile of %u fragments", mt);
}
#undef VX_PS_CASE

}  // namespace

bool gemm_ps_eligible(const GemmArgs &a) {
    if (a.T == 0 || a.T > kPiece || a.x_block) return false;
    if (a.epi == GEPI_SWIGLU) return a.o_tiled && a.oh && !a.seg[0].out && a.seg[0].rows % 32u == 0u && a.ldp % 32u == 0u;
    if (a.epi == GEPI_STORE) return a.ksplit <= 1u || a.split_store;
    return a.ksplit <= 1u || a.ws != nullptr;
}

// Called by launch_gemm_pf with arguments it has validated; sets the tiling fields.
int launch_gemm_ps(hipStream_t s, GemmArgs a) {
    const uint32_t kRows = a.epi == GEPI_SWIGLU ? 64u : 32u;
    uint32_t tiles = 0;
    if (a.epi == GEPI_SWIGLU) {
        tiles = (2u * a.seg[0].rows + kRows - 1u) / kRows;
    } else {
        for (uint32_t i = 0; i < a.nseg; ++i) {
            a.seg[i].tile0 = tiles;
            tiles += (a.seg[i].rows + kRows - 1u) / kRows;
        }
    }
    if (a.ksplit == 0) a.ksplit = 1;
    if (a.ksplit > a.K / 32u) a.ksplit = a.K / 32u;
    a.ntn = tiles;
    a.ntm = 1;
    const uint64_t grid = (uint64_t)tiles * a.ksplit;
    if (grid == 0) return VX_OK;
    if (grid > 0x7fffffffull) return fail(VX_ERR_UNSUPPORTED, "short prefill gemm: grid too large");
#define VX_PS_KIND(WKV, EP) \
    if (a.wk == WKV && a.epi == EP) return launch_ps<WKV, EP>(s, a, (uint32_t)grid);
    VX_PS_KIND(WT_Q8, GEPI_STORE)
    VX_PS_KIND(WT_Q8, GEPI_RESIDUAL)
    VX_PS_KIND(WT_Q8, GEPI_SWIGLU)
    VX_PS_KIND(WT_F16, GEPI_STORE)
    VX_PS_KIND(WT_F16, GEPI_RESIDUAL)
    VX_PS_KIND(WT_F16, GEPI_SWIGLU)
#undef VX_PS_KIND
    return fail(VX_ERR_UNSUPPORTED, "gemm: epilogue %u", a.epi);
}

// F16, no split: 32-row tiles of 64 tokens, and smaller ones while they leave CUs idle.
// The AudioVAE's up-convolutions and 1x1 convolutions of a 4-frame patch, against k_gemm's
// tiles with atomic sums into a cleared output (two launches): 21 + 2 -> 14.7 us for the
// 67 MB of the first (13 us at the copy rate), 11 + 2 -> 9.4 for the second, 9 -> 7 for a
// 1x1 convolution.
int launch_gemm_ps_tiles(hipStream_t s, GemmArgs a) {
    if (a.wk != WT_F16 || a.nseg != 1 || a.ksplit > 1u || a.T == 0 || a.K % 32u || !a.seg[0].pq || !a.xh || !a.xl ||
        !a.seg[0].out || !a.seg[0].rows)
        return fail(VX_ERR_INVALID_ARG, "short gemm: one F16 matrix in the prefill layout, K %% 32, no split");
    if ((a.epi == GEPI_STORE) != (a.x_block != 0u) || (a.epi != GEPI_STORE && a.epi != GEPI_RESIDUAL))
        return fail(VX_ERR_UNSUPPORTED, "short gemm: block-major store or tiled residual");
    if (a.pre && (a.epi != GEPI_RESIDUAL || !a.oh || !a.ol || a.o_block % 64u || a.o_block / 64u <= a.T ||
                  a.seg[0].rows % 32u || a.seg[0].ldo != a.seg[0].rows))
        return fail(VX_ERR_INVALID_ARG, "short gemm: planes of %u rows, block %u", a.T, a.o_block);
    uint32_t mt = a.T <= 16u ? 1u : a.T <= 32u ? 2u : 4u, nf = 2;
    const uint64_t ntn = (a.seg[0].rows + 31u) / 32u;
    if (a.pre || ntn * ((a.T + 16u * mt - 1u) / (16u * mt)) <= 96u) nf = 1;
    a.ksplit = 1;
    a.seg[0].tile0 = 0;
    a.ntn = (a.seg[0].rows + 16u * nf - 1u) / (16u * nf);
    a.ntm = (a.T + 16u * mt - 1u) / (16u * mt);
    const uint64_t grid = (uint64_t)a.ntn * a.ntm;
    if (grid > 0x7fffffffull) return fail(VX_ERR_UNSUPPORTED, "short gemm: grid too large");
    if (a.epi == GEPI_STORE)
        return nf == 1 ? launch_ps_tiles<GEPI_STORE, 1, true>(s, a, (uint32_t)grid, mt)
                       : launch_ps_tiles<GEPI_STORE, 2, true>(s, a, (uint32_t)grid, mt);
    return nf == 1 ? launch_ps_tiles<GEPI_RESIDUAL, 1, false>(s, a, (uint32_t)grid, mt)
                   : launch_ps_tiles<GEPI_RESIDUAL, 2, false>(s, a, (uint32_t)grid, mt);
}

}  // namespace vx
