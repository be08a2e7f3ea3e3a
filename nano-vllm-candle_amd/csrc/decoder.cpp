// Shared host half of the decoders built from layer descriptions: see decoder.h.
#include "decoder.h"
#include "hybrid.h"

#include <algorithm>

// Up to 16 rows a short K is the row kernels', whose activation needs no launch of its own.  A product of 1 / 16 rows, us, streamed and by rows: 9216 x 2048 9.9 / 10.4 and 11.0 / 13.2, 16384 x 1024
// 9.4 / 9.7 and 8.6 / 9.7; 9216 x 3072 13.3 / 14.2 and 17.3 / 25.0, 6144 x 4096 11.5 / 12.7 and 15.3 / 25.1, 24576 x 4096 34 / 37 and 50 / 62.  A step of layers 4096 wide, us, 1, 8 and 16 rows, before
// and with it: three of gopunex 494 538 570 and 409 424 445, two of berevik 317 347 369 and 290 291 300, two scans of tafopel 378 417 448 and 329 345 356.
static bool row_wins(const PackedW& w, int epi, int R) { return R <= 16 && w.K <= 2048 && gemm_rowpar_ok(w.N, w.K, epi, R); }
// y = x.W^T left as f32 slabs
ProductPlan plan_product(const nvllm_model* m, int R, const PackedW& w) {
    ProductPlan p;
    const size_t one = (size_t)R * w.N;
    p.max_split = (int)std::max<size_t>(1, std::min<size_t>(8, m->slab_floats / one));
    const int tmin = m->opt_tile_min_wgs;
    if (tmin > 0 && R > kRowMaxRows) {
        const int ks = gemm_tile_splits(R, w.N, w.K, tmin, std::min(p.max_split, R <= 512 ? 8 : 4));
        if (ks > 0) { p.kind = P_TILE; p.packed = 1; p.max_split = std::min(p.max_split, R <= 512 ? 8 : 4); return p; }
    }
    if (gemm_streams(m, w, R) && !row_wins(w, 2, R)) { p.kind = P_STREAM; p.packed = 1; return p; }
    if (R <= kRowMaxRows && gemm_rowpar_ok(w.N, w.K, 2, R) && (size_t)gemm_rowpar_splits(w.N, w.K, 2, R) * one <= m->slab_floats) {
        p.kind = P_ROW;
        p.packed = R >= kPackedMinRows && gemm_rowdir_ok(w.N, w.K, 2, R);
    }
    return p;
}
int run_product(nvllm_model* m, const ProductPlan& p, const bf16_bits* xh, const bf16_bits* xl, const PackedW& w, float* out, int R, int* n_slabs) {
    hipStream_t s = m->ctx->stream;
    if (p.kind == P_TILE) {
        PROF(m, PROF_GEMM, launch_gemm_tile(xh, xl, w, R, 0, out, nullptr, nullptr, 0, m->opt_tile_min_wgs, p.max_split, n_slabs, s));
        ++m->tile_launches;
    } else if (p.kind == P_STREAM) {
        PROF(m, PROF_GEMM, launch_gemm_stream(xh, xl, w.K, w, out, R, p.packed, s));
        *n_slabs = gemm_stream_splits(R, w.N, w.K);
    } else if (p.kind == P_ROW) {
        RowParArgs a;
        a.xh = xh; a.xl = xl; a.ldx = w.K; a.out = out; a.M = R; a.x_packed = p.packed;
        PROF(m, PROF_GEMM, launch_gemm_rowpar(a, w, 2, s));
        *n_slabs = gemm_rowpar_splits(w.N, w.K, 2, R);
    } else {
        GemmPlan g = plan_gemm(R, w.N, w.K, p.max_split);
        PROF(m, PROF_GEMM, launch_gemm(g, xh, xl, w.K, w, out, R, s));
        *n_slabs = g.n_split;
    }
    return NVLLM_OK;
}

int run_two_products(nvllm_model* m, const ProductJob& a, const ProductJob& b, int R) {
    if (a.p.kind == P_ROW && b.p.kind == P_ROW && gemm_rowdir_two_ok(a.w, b.w, R)) {
        auto args = [&](const ProductJob& j) {
            RowParArgs r;
            r.xh = j.xh; r.xl = j.xl; r.ldx = j.w.K; r.out = j.out; r.M = R; r.x_packed = j.p.packed;
            return r;
        };
        PROF(m, PROF_GEMM, launch_gemm_rowdir_two(args(a), a.w, args(b), b.w, m->ctx->stream));
        ++m->two_launches;
        *a.n_slabs = *b.n_slabs = 1;
        return NVLLM_OK;
    }
    int rc = run_product(m, a.p, a.xh, a.xl, a.w, a.out, R, a.n_slabs);
    if (!rc) rc = run_product(m, b.p, b.xh, b.xl, b.w, b.out, R, b.n_slabs);
    return rc;
}

GluPlan plan_glu(const nvllm_model* m, int R, const PackedW& w, bool want_packed_out) {
    GluPlan g;
    const int tmin = m->opt_tile_min_wgs;
    if (tmin > 0 && R > kRowMaxRows && gemm_tile_ok(R, w.N, w.K, 2, tmin)) { g.kind = P_TILE; g.packed = 1; g.out_packed_ok = 1; return g; }
    if (R <= kRowMaxRows && gemm_rowpar_ok(w.N, w.K, 1, R) && !(R <= 16 && gemm_streams(m, w, R) && !row_wins(w, 1, R))) {
        g.kind = P_ROW;
        const bool dir = gemm_rowdir_ok(w.N, w.K, 1, R);
        g.packed = R >= kPackedMinRows && dir;
        g.out_packed_ok = dir;
        return g;
    }
    if ((R > 16 ? gemm_stream_splits(R, w.N, w.K) > 0 : gemm_streams(m, w, R)) || want_packed_out) {
        g.kind = P_STREAM;
        g.slabs = plan_product(m, R, w);
        g.packed = g.slabs.packed;
        g.out_packed_ok = 1;
    }
    return g;
}
int run_glu(nvllm_model* m, const GluPlan& g, const bf16_bits* xh, const bf16_bits* xl, const PackedW& w, int R, const GluSpec& spec,
                   bf16_bits* oh, bf16_bits* ol, int out_packed) {
    hipStream_t s = m->ctx->stream;
    if (g.kind == P_TILE) {
        PROF(m, PROF_GEMM, launch_gemm_tile(xh, xl, w, R, 2, nullptr, oh, ol, out_packed, m->opt_tile_min_wgs, 1, nullptr, s, spec));
        ++m->tile_launches;
    } else if (g.kind == P_ROW) {
        RowParArgs a;
        a.xh = xh; a.xl = xl; a.ldx = w.K; a.oh = oh; a.ol = ol; a.M = R; a.x_packed = g.packed; a.o_packed = out_packed; a.glu = spec;
        PROF(m, PROF_GEMM, launch_gemm_rowpar(a, w, 1, s));
    } else if (g.kind == P_STREAM) {
        int ns = 1;
        int rc = run_product(m, g.slabs, xh, xl, w, m->slabs, R, &ns);
        if (rc) return rc;
        PROF(m, PROF_SILU, launch_silu_mul_interleaved(m->slabs, ns, (int64_t)R * w.N, R, w.N / 2, oh, ol, out_packed, s, spec));
    } else {
        GemmPlan p = plan_gemm_swiglu(R, w.N, w.K);
        PROF(m, PROF_GEMM, launch_gemm_swiglu(p, xh, xl, w.K, w, R, oh, ol, nullptr, s, spec));
    }
    return NVLLM_OK;
}

int run_act(nvllm_model* m, const ProductPlan& p, nvllm::Act act, const bf16_bits* xh, const bf16_bits* xl, const PackedW& w, int R, bf16_bits* oh, bf16_bits* ol, int out_packed) {
    hipStream_t s = m->ctx->stream;
    if (p.kind == P_TILE && gemm_tile_act_ok(R, w.N, w.K, act, m->opt_tile_min_wgs, p.max_split)) {
        PROF(m, PROF_GEMM, launch_gemm_tile(xh, xl, w, R, 4 + act, nullptr, oh, ol, out_packed, m->opt_tile_min_wgs, 1, nullptr, s));
        ++m->tile_launches;
    } else if (p.kind == P_ROW && gemm_rowdir_ok(w.N, w.K, 3 + act, R)) {
        RowParArgs a;
        a.xh = xh; a.xl = xl; a.ldx = w.K; a.oh = oh; a.ol = ol; a.M = R; a.x_packed = p.packed; a.o_packed = out_packed;
        PROF(m, PROF_GEMM, launch_gemm_rowpar(a, w, 3 + act, s));
    } else {
        int ns = 1, rc = run_product(m, p, xh, xl, w, m->slabs, R, &ns);
        if (rc) return rc;
        PROF(m, PROF_SILU, launch_act(act, m->slabs, ns, (int64_t)R * w.N, R, w.N, oh, ol, out_packed, s));
    }
    return NVLLM_OK;
}

// 32-bit product of row-major f32 rows
int exact_product(nvllm_model* m, const float* x, const PackedW& w, float* out, int R, int* n_slabs, int act) {
    HeadGemmArgs a;
    a.x = x; a.x_row = w.K; a.w = w.data; a.N = a.n_valid = w.N; a.K = w.K; a.M = R; a.exact = 1; a.y = out; a.y_row = w.N; a.act = act;
    if (n_slabs) {
        a.y_slab = (int64_t)R * w.N;
        a.splits = (int)std::max<int64_t>(1, std::min<int64_t>(exact_splits(R, w.N, w.K), (int64_t)m->slab_floats / a.y_slab));
        *n_slabs = a.splits;
    }
    PROF(m, PROF_GEMM, launch_head_gemm(a, m->ctx->stream));
    return NVLLM_OK;
}

int LastRows::alloc(nvllm_model* m, bool f32, size_t width0, size_t width1, int ldr) {
    nvllm_ctx* ctx = m->ctx;
    const size_t n = last_rows_cap(m), n16 = (n + 15) / 16 * 16, width[2] = {width0, width1};
    int rc = dmalloc(ctx, &m->last_resid, n * ldr);
    for (int i = 0; i < 2 && !rc; ++i) {
        if (!width[i]) continue;
        if (f32) { rc = dmalloc(ctx, &f[i], n * width[i]); continue; }
        for (bf16_bits** p : {&h[i], &l[i]}) {  // read in whole 16-row blocks
            if (!rc) rc = dmalloc(ctx, p, n16 * width[i]);
            if (!rc) HIPCHK(ctx, hipMemsetAsync(*p, 0, n16 * width[i] * 2, ctx->stream));
        }
    }
    return rc;
}
void LastRows::free() {
    for (int i = 0; i < 2; ++i) {
        for (void* p : {(void*)h[i], (void*)l[i], (void*)f[i]}) if (p) (void)hipFree(p);
        h[i] = l[i] = nullptr;
        f[i] = nullptr;
    }
}
GatherSet LastRows::set(int i, const bf16_bits* xh, const bf16_bits* xl, const float* x, int ld, int in_packed, int out_packed) const {
    GatherSet g;
    g.h = xh; g.l = xl; g.f = x; g.oh = h[i]; g.ol = l[i]; g.of = f[i]; g.ld = ld; g.in_packed = in_packed; g.out_packed = out_packed;
    return g;
}

int output_head(nvllm_model* m, const PackedW& head, int Kw, int Vp, const float* y, float cap, int n_last, int logits_row0) {
    nvllm_ctx* ctx = m->ctx;
    hipStream_t s = ctx->stream;
    const int tps = ctx->tp_size;
    uint32_t* ids_dst = tps == 1 ? m->d_next + logits_row0 : m->d_next + m->cur_n + (size_t)ctx->tp_rank * m->cur_n + logits_row0;
    float* val_dst = tps == 1 ? nullptr : m->d_maxval + (size_t)ctx->tp_rank * m->cur_n + logits_row0;
    float* lg = m->logits + (size_t)logits_row0 * m->V_l;
    if (!y && m->V_l % 16 == 0) {
        RowNorm rn;
        rn.softcap = cap;
        GemmPlan pl = plan_lmhead(n_last, m->V_l, Kw);
        PROF(m, PROF_LMHEAD, launch_gemm_argmax(pl, m->xh, m->xl, Kw, head, m->want_logits ? lg : nullptr, n_last, m->part_val, m->part_idx, &rn, s));
        if (!m->want_ids) return NVLLM_OK;
        const int parts = gemm_argmax_parts(pl, m->V_l);
        if (pl.lm_nt > 0) HIPCHK(ctx, launch_argmax_rows(m->part_val, m->part_idx, parts, n_last, ids_dst, val_dst, s));
        else HIPCHK(ctx, launch_argmax_parts(m->part_val, m->part_idx, parts, n_last, m->argmax_scratch, ids_dst, val_dst, s));
        return NVLLM_OK;
    }
    int ns = 1, rc = NVLLM_OK;
    if (y && !(cap > 0.f)) {  // the product is the logits: a launch of 5 us fewer for 16 rows of 32768
        HeadGemmArgs a;
        a.x = y; a.x_row = head.K; a.w = head.data; a.N = head.N; a.n_valid = m->V_l; a.K = head.K; a.M = n_last; a.exact = 1; a.y = lg; a.y_row = m->V_l;
        PROF(m, PROF_LMHEAD, launch_head_gemm(a, s));
        if (m->want_ids) HIPCHK(ctx, launch_argmax(lg, n_last, m->V_l, m->V_l, ids_dst, val_dst, s));
        return NVLLM_OK;
    }
    if (y) rc = exact_product(m, y, head, m->slabs, n_last);
    else {
        ProductPlan ph;  // row-major planes, one slab
        rc = run_product(m, ph, m->xh, m->xl, head, m->slabs, n_last, &ns);
    }
    if (rc) return rc;
    HIPCHK(ctx, launch_logits_finish(m->slabs, ns, (int64_t)n_last * Vp, Vp, n_last, m->V_l, cap, lg, m->V_l, s));
    if (m->want_ids) HIPCHK(ctx, launch_argmax(lg, n_last, m->V_l, m->V_l, ids_dst, val_dst, s));
    return NVLLM_OK;
}
