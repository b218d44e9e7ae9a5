// The benchmark-config forward over the compacted token stream, enqueued by one call: offsets, tokenizer, blocks, heads.
// Two forms of a block: attention + one kernel for the rest (block_tail.h) where images are given, else one kernel per op.
// The host's share of a forward is this function's launches; composed in Python from the same entry points it was 270 us per
// forward at two layers, which is what a small batch then took.
#include "cfg_env_f32.h"
#include "cfg_env_rows.h"
#include "linear_args.h"

namespace {

struct Bump {
    char* p; size_t used = 0;
    void* take(size_t n) { void* r = p ? p + used : nullptr; used += (n + 255) & ~(size_t)255; return r; }
};

// d = 256 keeps the residual stream fp32 between the kernels in either form: the block-stack kernel, which smaller batches of
// the model take, keeps it in fp32 registers, and no batch size lowers the precision
bool stream_f32(const bsrl_cfg_desc& d) { return d.d == 256 && d.dtype != BSRL_F32; }

struct RowsPlan {
    int32_t* noff; void *x0, *x1, *h, *q, *att, *hid, *lead; size_t bytes;
    u16* ex1; float* epart;                          // the few-envs form (in the place of the others)
    RowsPlan(const bsrl_cfg_desc& d, int64_t B, bool tail, char* ws) {
        const size_t es = d.dtype == BSRL_F32 ? 4 : 2, R = (size_t)B * d.T, D = d.d, xs = stream_f32(d) ? 4 : es;
        Bump b{ws};
        noff = static_cast<int32_t*>(b.take((B + 1) * 4));
        x0 = b.take(R * D * xs);
        x1 = b.take(R * D * xs);
        q = b.take(R * 3 * D * es);
        att = b.take(R * D * es);
        h = b.take((tail ? (size_t)B : R) * D * es);
        hid = b.take(tail ? 0 : R * d.ffn * es);
        lead = b.take((size_t)B * D * es);
        bytes = b.used;
        if (!tail && bsrl_cfg_env_rows_pack_size(&d) > 0) {
            Bump e{ws};
            e.take((B + 1) * 4);
            ex1 = static_cast<u16*>(e.take((R + B) * D * 2));
            epart = static_cast<float*>(e.take(4 * R * D * 4));
            if (e.used > bytes) bytes = e.used;
        }
    }
};

bool rows_desc_ok(const bsrl_cfg_desc* d) {
    return d && d->n_layers >= 1 && d->n_layers <= BSRL_MAX_LAYERS && d->n_heads >= 1 && d->d > 0 && d->d % d->n_heads == 0 && d->ffn > 0 &&
           d->T >= 1 && d->T <= BSRL_MAX_T && d->n_gears >= 1 && d->prop_dim >= 1 && d->obj_dim >= 1;
}

}  // namespace

extern "C" int64_t bsrl_cfg_rows_workspace_size(const bsrl_cfg_desc* d, int64_t B, int tail) {
    if (!rows_desc_ok(d) || B < 0) return 0;
    return (int64_t)RowsPlan(*d, B, tail != 0, nullptr).bytes;
}

extern "C" int64_t bsrl_cfg_rows_pack_size(const bsrl_cfg_desc* d) {
    return !rows_desc_ok(d) ? 0 : d->dtype == BSRL_F32 ? bsrl_cfg_env_f32_pack_size(d) : bsrl_cfg_env_rows_pack_size(d);
}

extern "C" int bsrl_cfg_rows_pack(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w, void* img, bsrl_stream stream) {
    if (!rows_desc_ok(d) || !w || !img) BSRL_FAIL(BSRL_EINVAL, "bsrl_cfg_rows_pack: null pointer or bad shape");
    if (bsrl_cfg_rows_pack_size(d) == 0) return BSRL_UNSUPPORTED;
    if (!bsrl_aligned(img, 16)) BSRL_FAIL(BSRL_EINVAL, "bsrl_cfg_rows_pack: image must be 16-byte aligned");
    return d->dtype == BSRL_F32 ? bsrl_cfg_env_f32_pack(d, w, img, static_cast<hipStream_t>(stream)) : bsrl_cfg_env_rows_pack(d, w, img, static_cast<hipStream_t>(stream));
}

extern "C" int bsrl_cfg_rows_forward(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w, const void* obs, int64_t obs_ld,
                                     int obs_dtype, const int32_t* n_valid, float* logits, float* value, int64_t B, int prune,
                                     void* workspace, int64_t workspace_bytes, bsrl_stream stream) {
    if (!rows_desc_ok(d) || !w || !obs || !logits || !value) BSRL_FAIL(BSRL_EINVAL, "bsrl_cfg_rows_forward: null pointer or bad shape");
    if (B < 0 || B * d->T > 0x7fffffffLL) BSRL_FAIL(BSRL_EINVAL, "bsrl_cfg_rows_forward: bad batch");
    if (B == 0) return BSRL_OK;
    const bool tail = w->blk[0].tail_img != nullptr;
    RowsPlan p(*d, B, tail, static_cast<char*>(workspace));
    if (!workspace || workspace_bytes < (int64_t)p.bytes || !bsrl_aligned(workspace, 16)) BSRL_FAIL(BSRL_EINVAL, "bsrl_cfg_rows_forward: workspace too small");
    const int64_t D = d->d, F = d->ffn, R = B * d->T, H = d->n_heads, dh = D / H, opt = d->T - 1;
    const int dt = d->dtype, es = dt == BSRL_F32 ? 4 : 2, L = d->n_layers, act = d->act;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int32_t* extra = p.noff + B;
    int rc;
    // One launch, an env's rows in LDS.  It computes all of an env's token slots, the launches below the attendable ones alone: with half of
    // them masked these win from about ten envs per CU on (us, one launch | launches: 256 envs 42 | 107, 2048 230 | 255, 4096 455 | 394;
    // no mask: 256 envs 42 | 113, 4096 456 | 554, 16384 1803 | 2041)
    if (dt == BSRL_F32 && obs_dtype == BSRL_F32 && prune && w->lead_img && bsrl_aligned(w->lead_img, 16) && bsrl_cfg_env_f32_pack_size(d) > 0 &&
        (!n_valid || B <= 10 * (int64_t)bsrl_cus())) {
        const CfgEnvF32Args e{*w, static_cast<const float*>(obs), obs_ld, n_valid, logits, value, (int)B, L, d->T, (int)(29 * d->n_gears + 1), d->final_ln, d->prop_dim, d->obj_dim};
        if (bsrl_cfg_env_f32(d, e, st)) {
            BSRL_CHECK_LAUNCH("bsrl_cfg_rows_forward");
            return BSRL_OK;
        }
    }
#define STEP(call) do { if ((rc = (call)) != BSRL_OK) return rc; } while (0)
    auto at = [&](const void* q, int64_t elems) { return static_cast<const char*>(q) + elems * es; };
    // y = act(x W^T + b) (+ res) on rows [+ *extra] rows; res_f32, y_f32: that operand is fp32
    auto linear = [&](const void* x, int64_t ldx, const void* W, const float* b, const void* res, void* y, int64_t K, int64_t M, int a_, bool all,
                      bool res_f32 = false, bool y_f32 = false) {
        LinArgs a{x, ldx, W, b, res, D, y, M, nullptr, 0, 0, all ? R : B, (int)K, (int)M, y_f32, 0, 0, nullptr, 0};
        a.res_f32 = res_f32;
        if (all) { a.extra = extra; a.base = B; }
        if (!bsrl_linear_small(a, a_, dt, st)) return (int)BSRL_UNSUPPORTED;
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) BSRL_FAIL(BSRL_ELAUNCH, "bsrl_cfg_rows_forward: %s", hipGetErrorString(e));
        return (int)BSRL_OK;
    };
    STEP(bsrl_token_offsets(n_valid, B, opt, p.noff, stream));
    if (!tail && prune && bsrl_cfg_env_rows_ok(d, w)) {
        const CfgEnvRowsArgs e{*w, obs, obs_ld, p.noff, p.ex1, p.epart, logits, value, (int)B, L, d->T, (int)(29 * d->n_gears + 1), d->final_ln, d->prop_dim, d->obj_dim,
                               obs_dtype == BSRL_F32};
        return bsrl_cfg_env_rows(d, e, st);
    }
    STEP(bsrl_cfg_tokens(obs, obs_ld, obs_dtype, w->prop_w, w->prop_b, w->obj_w, w->obj_b, p.noff, p.x0, B, D, d->prop_dim, d->obj_dim, dt, stream));
    const float eps = 1e-5f;
    void *x = p.x0, *xn = p.x1;
    const bool f32s = stream_f32(*d);
    auto next_cols = [&](int i) { return prune && i + 1 == L ? 2 * D : 3 * D; };      // the final block projects keys and values only
    if (tail) STEP(bsrl_block_tail(w->lead_img, nullptr, x, nullptr, nullptr, 0.f, w->blk[0].ln_attn_w, w->blk[0].ln_attn_b, eps, nullptr,
                                   next_cols(0) == 2 * D ? p.h : nullptr, B, p.q, next_cols(0), B, extra, R - B, D, 0, act, dt, 0, stream));
    for (int i = 0; i < L; ++i) {
        const auto& k = w->blk[i];
        const bool pruned = prune && i + 1 == L, xf = f32s && i > 0, last = i + 1 == L;      // xf: this block's rows come in as fp32
        const int64_t qn = next_cols(i);
        if (!tail) {
            STEP(bsrl_ln_rows(x, D, k.ln_attn_w, k.ln_attn_b, p.h, D, nullptr, nullptr, B, extra, R, D, eps, dt, stream, xf));
            STEP(linear(p.h, D, at(k.qkv_w, (3 * D - qn) * D), k.qkv_b + (3 * D - qn), nullptr, p.q, D, qn, BSRL_ACT_NONE, true));
        }
        const void *qp = p.q, *kp = at(p.q, qn - 2 * D), *vp = at(p.q, qn - D);
        int64_t qld = qn;
        if (pruned) {      // the query of token 0 alone
            if (tail) STEP(bsrl_linear(p.h, D, k.qkv_w, k.qkv_b, nullptr, 0, p.lead, D, nullptr, 0, 0, B, D, D, BSRL_ACT_NONE, dt, dt, stream));
            else STEP(linear(p.h, D, k.qkv_w, k.qkv_b, nullptr, p.lead, D, D, BSRL_ACT_NONE, false));
            qp = p.lead; qld = D;
        }
        STEP(bsrl_attn_ragged(qp, qld, kp, qn, vp, qn, p.noff, nullptr, p.att, D, B, 1, opt, pruned, H, dh, dt, stream));
        const int64_t extra_max = pruned ? 0 : R - B;
        const int32_t* ex = pruned ? nullptr : extra;
        if (tail) {
            const int64_t nn = last ? 0 : next_cols(i + 1);
            const auto* nk = last ? nullptr : &w->blk[i + 1];
            const int x_f32 = (xf ? 1 : 0) | (f32s && !last ? 2 : 0);
            STEP(bsrl_block_tail(k.tail_img, p.att, x, k.ln_ffn_w, k.ln_ffn_b, eps, nk ? nk->ln_attn_w : nullptr, nk ? nk->ln_attn_b : nullptr, eps,
                                 xn, nn == 2 * D ? p.h : nullptr, B, nn ? p.q : nullptr, nn, B, ex, extra_max, D, F, act, dt, x_f32, stream));
            void* t = x; x = xn; xn = t;
        } else {
            STEP(linear(p.att, D, k.out_w, k.out_b, x, xn, D, D, BSRL_ACT_NONE, !pruned, xf, f32s));
            STEP(bsrl_ln_rows(xn, D, k.ln_ffn_w, k.ln_ffn_b, p.h, D, nullptr, nullptr, B, ex, B + extra_max, D, eps, dt, stream, f32s));
            STEP(linear(p.h, D, k.w0, k.b0, nullptr, p.hid, D, F, act, !pruned));
            STEP(linear(p.hid, F, k.w2, k.b2, xn, x, F, D, BSRL_ACT_NONE, !pruned, f32s, f32s && !last));
        }
    }
    if (d->final_ln) {
        STEP(bsrl_ln_fwd(x, w->final_ln_w, w->final_ln_b, p.lead, nullptr, nullptr, B, D, eps, dt, stream));
        x = p.lead;
    }
    const int64_t n_log = 29 * (int64_t)d->n_gears;
    STEP(bsrl_linear(x, D, w->heads_w, w->heads_b, nullptr, 0, logits, n_log, value, 1, n_log, B, D, n_log + 1, BSRL_ACT_NONE, dt, BSRL_F32, stream));
#undef STEP
    return BSRL_OK;
}
