// Token-batched prefill of a layer stack (the seq_* op family of
// local.rs:482-527 applied to a MiniCPM4-style decoder stack, with a causal mask
// and a position base), shared by the BaseLM (with RoPE) and the ResidualLM
// (without RoPE):
//   per layer over the rows of the residual stream h:
//     rmsnorm(h)*attn_norm -> f16 hi/lo planes        (k_seq_rmsnorm)
//     q|k|v = planes . Wq|Wk|Wv                       (GEMM, split-K)
//     RoPE at pos0+t (or none), K/V rows -> f16 cache, q planes  (k_prefill_rope)
//     causal attention over cache keys 0..pos0+t       (k_prefill_attn)
//     h += scale * Wo . attn                           (GEMM, residual)
//     rmsnorm(h)*ffn_norm -> planes                    (k_seq_rmsnorm)
//     act = silu(Wg . n) * (Wu . n) -> planes          (GEMM, SwiGLU)
//     h += scale * Wdown . act                         (GEMM, residual)
// The GEMM is k_gemm_pf over weights in the prefill layout (k_gemm_ps below 128 rows),
// k_gemm where the engine has none.
// Row t computes what the decode step computes at position pos0 + t: the same
// KV-cache rows and the same residual stream, to rounding.
#include <algorithm>
#include <type_traits>

#include "vx_internal.h"

namespace vx {

namespace {

// Split-K factor for a projection of n_tiles 128-row tiles and tt-token tiles:
// as many workgroups as fit one per CU (rounded down: a second workgroup on a CU
// runs at well under twice one's throughput, so the CUs that hold two would set
// the time; measured on MI355X, rounding up instead made the T = 384 prefill 5%
// slower, T = 256 and 512 2%), at least four 32-column blocks per split.
uint32_t pick_split(const vx_ctx *ctx, uint32_t tt, uint32_t n_tiles, uint32_t T, uint32_t K) {
    const uint32_t tiles = n_tiles * ((T + tt - 1u) / tt);
    const uint32_t cus = ctx->props.multiProcessorCount > 0 ? (uint32_t)ctx->props.multiProcessorCount : 256u;
    uint32_t ks = std::max<uint32_t>(1u, cus / tiles);
    ks = std::min<uint32_t>(ks, tt > 64u ? 8u : 4u);
    ks = std::min<uint32_t>(ks, std::max<uint32_t>(1u, K / 128u));
    return std::max<uint32_t>(ks, 1u);
}

// The same below a whole token tile (k_gemm_ps, 32-row tiles): every workgroup reads
// all of X, so one per CU (two were 10% slower at 37 rows), four blocks or more each.
uint32_t pick_split_short(const vx_ctx *ctx, uint32_t n_tiles, uint32_t K) {
    const uint32_t cus = ctx->props.multiProcessorCount > 0 ? (uint32_t)ctx->props.multiProcessorCount : 256u;
    return std::max<uint32_t>(1u, std::min({cus / n_tiles, K / 128u, kPrefillMaxSplit}));
}

// Rows from one partial slab to the next, at least. Slabs close together slow the GEMM
// that writes them and the one after it: four Q8_0 layers at 200 / 256 / 384 rows took
// 474 / 502 / 617 us with slabs of exactly those rows (and 64 to 2048 floats more), 459 /
// 488 / 610 with 512 rows, 455 / 473 / 602 with 1000 or 1024.
constexpr uint32_t kSlabRows = 1024u;

GemmSeg gemm_seg(const WRef &w, uint32_t rows, float *out, uint32_t ldo) {
    GemmSeg g;
    if (w.wt == WT_Q8) {
        g.qs = static_cast<const int8_t *>(w.ptr);
        g.d = w.d;
    } else {
        g.w = static_cast<const __half *>(w.ptr);
    }
    g.rows = rows;
    g.out = out;
    g.ldo = ldo;
    return g;
}

}  // namespace

int prefill_stack_check(const PrefillStack &p) {
    for (uint32_t l = 0; l < p.n_layers; ++l) {
        const StackLayer &L = p.layers[l];
        const WRef *ws[] = {&L.q, &L.k, &L.v, &L.o, &L.gate, &L.up, &L.down};
        for (const WRef *w : ws) {
            if (w->wt == WT_Q8 && !w->ptr)
                return fail(VX_ERR_UNSUPPORTED,
                            "batched prefill needs Q8_0 row widths that are multiples of 1024 (layer %u)", l);
            if (w->wt == WT_F16 && (w->cols % 128u))
                return fail(VX_ERR_UNSUPPORTED, "batched prefill needs F16 row widths that are multiples of 128");
            if (w->wt == WT_F32) return fail(VX_ERR_UNSUPPORTED, "batched prefill has no F32 projection path");
        }
    }
    if (p.head_dim != 64u && p.head_dim != 128u)
        return fail(VX_ERR_UNSUPPORTED, "batched prefill attention needs head_dim 64 or 128");
    const uint32_t qpk = p.q_heads / p.kv_heads;
    if (qpk != 1u && qpk != 2u && qpk != 4u && qpk != 8u)
        return fail(VX_ERR_UNSUPPORTED, "batched prefill attention needs 1, 2, 4 or 8 query heads per KV head");
    if (p.rope && !p.rope_factors) return fail(VX_ERR_INVALID_ARG, "batched prefill with RoPE needs its factors");
    return VX_OK;
}

int prefill_stack_weights(vx_ctx *ctx, const StackLayer *layers, uint32_t n_layers, uint32_t nH, uint32_t nF,
                          uint32_t nKV, std::vector<StackPrefillWeights> *pw, vx_buf **arena) {
    pw->clear();
    if (!n_layers || nH % 32u || nF % 32u) return VX_OK;
    const uint32_t wt = layers[0].q.wt;
    for (uint32_t l = 0; l < n_layers; ++l) {
        const StackLayer &L = layers[l];
        for (const WRef *w : {&L.q, &L.k, &L.v, &L.o, &L.gate, &L.up, &L.down})
            if (w->wt != wt || (wt == WT_Q8 ? w->dtype != VX_DTYPE_Q8_0 || !w->raw
                                            : wt != WT_F16 || !w->ptr || ((uintptr_t)w->ptr & 15u)))
                return VX_OK;
    }
    const uint64_t per_layer = prefill_matrix_bytes(wt, nH, nH) + 2u * prefill_matrix_bytes(wt, nKV, nH) +
                               prefill_matrix_bytes(wt, nH, nH) + prefill_matrix_bytes(wt, 2u * nF, nH) +
                               prefill_matrix_bytes(wt, nH, nF) + 6u * 256u;
    const int st_alloc = vx_alloc(ctx, per_layer * n_layers, arena);
    if (st_alloc == VX_ERR_OOM && wt == WT_F16) return VX_OK;   // the general GEMM reads the model's own rows
    VX_CHECK(st_alloc);
    uint8_t *cur = static_cast<uint8_t *>((*arena)->ptr);
    hipStream_t s = ctx->stream;
    auto place = [&](PrefillMatrix &pm, const WRef &w0, const WRef *w1, uint32_t rows, uint32_t K) {
        const uint32_t rows_out = w1 ? 2u * rows : rows;
        pm.rows_pad = (rows_out + 127u) / 128u * 128u;
        pm.q = reinterpret_cast<int8_t *>(cur);
        pm.d = wt == WT_Q8 ? reinterpret_cast<float *>(cur + (uint64_t)pm.rows_pad * K) : nullptr;
        cur += (prefill_matrix_bytes(wt, rows_out, K) + 255u) / 256u * 256u;
        return wt == WT_Q8 ? launch_repack_prefill(s, w0.raw, w0.raw_offset, w1 ? w1->raw_offset : 0u, rows, K,
                                                   w1 ? 1 : 0, pm.q, pm.d)
                           : launch_repack_prefill_f16(s, static_cast<const __half *>(w0.ptr),
                                                       w1 ? static_cast<const __half *>(w1->ptr) : nullptr, rows, K,
                                                       pm.q);
    };
    pw->resize(n_layers);
    for (uint32_t l = 0; l < n_layers; ++l) {
        const StackLayer &L = layers[l];
        StackPrefillWeights &P = (*pw)[l];
        int st = VX_OK;
        if ((st = place(P.q, L.q, nullptr, nH, nH)) || (st = place(P.k, L.k, nullptr, nKV, nH)) ||
            (st = place(P.v, L.v, nullptr, nKV, nH)) || (st = place(P.o, L.o, nullptr, nH, nH)) ||
            (st = place(P.gu, L.gate, &L.up, nF, nH)) || (st = place(P.down, L.down, nullptr, nH, nF))) {
            pw->clear();
            vx_free(ctx, *arena);
            *arena = nullptr;
            return st;
        }
    }
    return VX_OK;
}

int prefill_stack_alloc(vx_ctx *ctx, uint32_t cap, uint32_t nH, uint32_t nF, uint32_t nKV, StackWork *w) {
    if (w->cap) return VX_OK;
    const uint64_t H = nH, F = nF, KV = nKV, T = cap;
    const uint64_t Tp = (T + 127u) / 128u * 128u;   // GEMM input planes: whole 128-token tiles
    // Split-K partials: of the residual projections ([split][T][H]) and of QKV
    // ([split][T][H + 2 KV]); the two uses never overlap in time. A split of more than one
    // has at most a workgroup per CU (pick_split), which bounds split * T above kSlabRows.
    const uint32_t cus = ctx->props.multiProcessorCount > 0 ? (uint32_t)ctx->props.multiProcessorCount : 256u;
    const uint64_t ws_rows =
        std::max<uint64_t>(kPrefillMaxSplit * kSlabRows, 128u * (uint64_t)cus / ((H + 127u) / 128u));
    // Stream-K SwiGLU: two tile parts per workgroup and a counter per workgroup
    // boundary, one workgroup per CU; the counters start at zero.
    w->sk_grid = cus / 8u * 8u;
    // One allocation: a new engine's first prefill waits for each.
    uint64_t bytes = 0;
    uint8_t *base = nullptr;
    auto lay = [&]() {
        bytes = 0;
        auto put = [&](auto *&ptr, uint64_t n) {
            ptr = reinterpret_cast<std::remove_reference_t<decltype(ptr)>>(base + bytes);
            bytes += (n + 255u) / 256u * 256u;
        };
        put(w->h, T * H * 4u);
        put(w->xh, Tp * H * 2u);
        put(w->xl, Tp * H * 2u);
        put(w->ah, Tp * F * 2u);
        put(w->al, Tp * F * 2u);
        put(w->qh, T * H * 2u);
        put(w->ql, T * H * 2u);
        put(w->q, T * H * 4u);
        put(w->k, T * KV * 4u);
        put(w->v, T * KV * 4u);
        put(w->ws, ws_rows * (H + 2u * KV) * 4u);
        put(w->rope, T * 64u * 8u);   // head_dim <= 128
        put(w->sk_ws, (uint64_t)w->sk_grid * 2u * kSkTileFloats * 4u);
        put(w->sk_cnt, (uint64_t)w->sk_grid * 4u);
    };
    lay();
    VX_CHECK(vx_alloc(ctx, bytes, &w->arena));
    base = static_cast<uint8_t *>(w->arena->ptr);
    lay();
    if (w->sk_grid) {
        const int st = launch_fill_u32(ctx->stream, w->sk_cnt, 0u, w->sk_grid);
        if (st != VX_OK) {
            prefill_stack_free(ctx, w);
            return st;
        }
    }
    w->cap = cap;
    return VX_OK;
}

void prefill_stack_free(vx_ctx *ctx, StackWork *w) {
    if (w->arena) vx_free(ctx, w->arena);
    *w = StackWork();
}

int enqueue_prefill_stack(const PrefillStack &p, uint32_t pos0, uint32_t T) {
    vx_ctx *ctx = p.ctx;
    hipStream_t s = ctx->stream;
    const StackWork &w = *p.work;
    const uint32_t nH = p.nH, nF = p.nF, nKV = p.nKV;
    if (T == 0 || T > w.cap) return fail(VX_ERR_INVALID_ARG, "prefill chunk of %u rows (capacity %u)", T, w.cap);
    // The prefill-layout weights and tiled planes go to the deep-pipelined GEMM from one
    // full 128-token tile up and to the short-chunk one below.
    const bool tiled = p.pw != nullptr;
    const bool is_short = tiled && T < gemm_pf_tile_tokens();
    const uint32_t tt = tiled ? gemm_pf_tile_tokens() : 64u;
    auto split = [&](uint32_t rows, uint32_t kv_rows, uint32_t K) {
        if (is_short) return pick_split_short(p.ctx, (rows + 31u) / 32u + 2u * ((kv_rows + 31u) / 32u), K);
        return pick_split(p.ctx, tt, (rows + 127u) / 128u + 2u * ((kv_rows + 127u) / 128u), T, K);
    };
    const uint32_t ks_qkv = split(nH, nKV, nH), ks_o = split(nH, 0, nH), ks_down = split(nH, 0, nF);
    // Split residual projections on the tiled path leave their partials in
    // the workspace; the next rmsnorm adds them to h (no atomics in the GEMM epilogue).
    const uint32_t slab = std::max(T, kSlabRows);
    const uint64_t ws_stride = (uint64_t)slab * nH;
    const bool ws_o = tiled && ks_o > 1, ws_down = tiled && ks_down > 1;
    // Split QKV on the tiled path stores its partials to the workspace as well (q, k, v
    // regions of one split, ws_qkv floats per split); the RoPE kernel sums them.
    const bool ws_qkv = tiled && ks_qkv > 1;
    const uint64_t ws_qkv_stride = (uint64_t)slab * (nH + 2u * nKV);
    float *const wq = w.ws, *const wk = wq + (size_t)slab * nH, *const wv = wk + (size_t)slab * nKV;
    float2 *const rope = p.rope ? w.rope : nullptr;
    for (uint32_t l = 0; l < p.n_layers; ++l) {
        const StackLayer &L = p.layers[l];
        {
            ProfSpan sp(ctx, "prefill.norm");
            SeqNormArgs n;
            n.h = w.h;
            n.ldh = nH;
            n.w = L.attn_norm;
            if (l > 0 && ws_down) {
                n.branch = w.ws;
                n.ldb = nH;
                n.nbranch = ks_down;
                n.branch_stride = ws_stride;
            }
            n.n = nH;
            n.eps = p.eps;
            n.yh = w.xh;
            n.yl = w.xl;
            n.ldp = nH;
            n.tiled = tiled ? 1u : 0u;
            if (ks_qkv > 1 && !ws_qkv) {
                n.zero[0] = w.q;
                n.zero_n[0] = nH;
                n.zero[1] = w.k;
                n.zero_n[1] = nKV;
                n.zero[2] = w.v;
                n.zero_n[2] = nKV;
            }
            VX_CHECK(launch_seq_rmsnorm(s, n, T));
        }
        {
            ProfSpan sp(ctx, "prefill.qkv");
            GemmArgs g;
            g.wk = L.q.wt;
            g.epi = GEPI_STORE;
            g.seg[0] = gemm_seg(L.q, nH, w.q, nH);
            g.seg[1] = gemm_seg(L.k, nKV, w.k, nKV);
            g.seg[2] = gemm_seg(L.v, nKV, w.v, nKV);
            if (tiled) {
                const StackPrefillWeights &P = p.pw[l];
                g.seg[0].pq = P.q.q;
                g.seg[0].pd = P.q.d;
                g.seg[1].pq = P.k.q;
                g.seg[1].pd = P.k.d;
                g.seg[2].pq = P.v.q;
                g.seg[2].pd = P.v.d;
                g.x_tiled = 1;
            }
            g.nseg = 3;
            g.K = nH;
            g.T = T;
            g.xh = w.xh;
            g.xl = w.xl;
            g.ldx = nH;
            g.ksplit = ks_qkv;
            if (ws_qkv) {
                g.seg[0].out = wq;
                g.seg[1].out = wk;
                g.seg[2].out = wv;
                g.split_store = 1;
                g.ws_stride = ws_qkv_stride;
            }
            VX_CHECK(launch_gemm(s, g));
        }
        {
            ProfSpan sp(ctx, "prefill.rope_store");
            SeqRopeArgs r;
            r.q = ws_qkv ? wq : w.q;
            r.k = ws_qkv ? wk : w.k;
            r.v = ws_qkv ? wv : w.v;
            if (ws_qkv) {
                r.nsplit = ks_qkv;
                r.split_stride = ws_qkv_stride;
            }
            r.ldq = nH;
            r.ldk = nKV;
            r.factors = p.rope_factors;
            r.pos_base = pos0;
            r.q_heads = p.q_heads;
            r.kv_heads = p.kv_heads;
            r.head_dim = p.head_dim;
            r.theta = p.theta;
            r.scaling = p.rope_scaling;
            r.qh = w.qh;
            r.ql = w.ql;
            r.ldqp = nH;
            r.kc = p.kc;
            r.vc = p.vc;
            r.layer = l;
            r.context = p.context;
            if (l == 0 && rope) VX_CHECK(launch_prefill_rope_table(s, r, T, rope));
            VX_CHECK(launch_prefill_rope(s, r, T, rope));
        }
        {
            ProfSpan sp(ctx, "prefill.attention");
            PrefillAttnArgs a;
            a.qh = w.qh;
            a.ql = w.ql;
            a.ldq = nH;
            a.kc = p.kc;
            a.vc = p.vc;
            a.layer = l;
            a.context = p.context;
            a.pos_base = pos0;
            a.T = T;
            a.q_heads = p.q_heads;
            a.kv_heads = p.kv_heads;
            a.head_dim = p.head_dim;
            a.oh = w.xh;
            a.ol = w.xl;
            a.ldo = nH;
            a.tiled = tiled ? 1u : 0u;
            VX_CHECK(launch_prefill_attn(s, a));
        }
        {
            ProfSpan sp(ctx, "prefill.attn_out");
            GemmArgs g;
            g.wk = L.o.wt;
            g.epi = GEPI_RESIDUAL;
            g.seg[0] = gemm_seg(L.o, nH, w.h, nH);
            if (tiled) {
                g.seg[0].pq = p.pw[l].o.q;
                g.seg[0].pd = p.pw[l].o.d;
                g.x_tiled = 1;
            }
            g.K = nH;
            g.T = T;
            g.xh = w.xh;
            g.xl = w.xl;
            g.ldx = nH;
            g.scale = p.residual_scale;
            g.ksplit = ks_o;
            if (ws_o) {
                g.ws = w.ws;
                g.ws_stride = ws_stride;
            }
            VX_CHECK(launch_gemm(s, g));
        }
        {
            ProfSpan sp(ctx, "prefill.norm");
            SeqNormArgs n;
            n.h = w.h;
            n.ldh = nH;
            n.w = L.ffn_norm;
            if (ws_o) {
                n.branch = w.ws;
                n.ldb = nH;
                n.nbranch = ks_o;
                n.branch_stride = ws_stride;
            }
            n.n = nH;
            n.eps = p.eps;
            n.yh = w.xh;
            n.yl = w.xl;
            n.ldp = nH;
            n.tiled = tiled ? 1u : 0u;
            VX_CHECK(launch_seq_rmsnorm(s, n, T));
        }
        {
            ProfSpan sp(ctx, "prefill.swiglu");
            GemmArgs g;
            g.wk = L.gate.wt;
            g.epi = GEPI_SWIGLU;
            g.seg[0] = gemm_seg(L.gate, nF, nullptr, 0);
            g.seg[1] = gemm_seg(L.up, nF, nullptr, 0);
            if (tiled) {
                g.seg[0].pq = p.pw[l].gu.q;   // gate and up interleaved
                g.seg[0].pd = p.pw[l].gu.d;
                g.x_tiled = 1;
                g.o_tiled = 1;
            }
            g.nseg = 2;
            g.K = nH;
            g.T = T;
            g.xh = w.xh;
            g.xl = w.xl;
            g.ldx = nH;
            g.oh = w.ah;
            g.ol = w.al;
            g.ldp = nF;
            if (tiled && w.sk_grid && p.schedule != VX_PREFILL_TILES) {
                g.sk_ws = w.sk_ws;
                g.sk_cnt = w.sk_cnt;
                g.sk_grid = w.sk_grid;
                g.sk_tail_first = p.schedule == VX_PREFILL_STREAMK_TAIL_FIRST ? 1u : 0u;
            }
            VX_CHECK(launch_gemm(s, g));
        }
        {
            ProfSpan sp(ctx, "prefill.down");
            GemmArgs g;
            g.wk = L.down.wt;
            g.epi = GEPI_RESIDUAL;
            g.seg[0] = gemm_seg(L.down, nH, w.h, nH);
            if (tiled) {
                g.seg[0].pq = p.pw[l].down.q;
                g.seg[0].pd = p.pw[l].down.d;
                g.x_tiled = 1;
            }
            g.K = nF;
            g.T = T;
            g.xh = w.ah;
            g.xl = w.al;
            g.ldx = nF;
            g.scale = p.residual_scale;
            g.ksplit = ks_down;
            if (ws_down) {
                g.ws = w.ws;
                g.ws_stride = ws_stride;
            }
            VX_CHECK(launch_gemm(s, g));
        }
    }
    if (ws_down) {   // the last layer's down partials
        ProfSpan sp(ctx, "prefill.norm");
        SeqNormArgs n;
        n.h = w.h;
        n.ldh = nH;
        n.n = nH;
        n.branch = w.ws;
        n.ldb = nH;
        n.nbranch = ks_down;
        n.branch_stride = ws_stride;
        VX_CHECK(launch_seq_rmsnorm(s, n, T));
    }
    return VX_OK;
}

}  // namespace vx
