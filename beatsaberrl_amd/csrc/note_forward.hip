// NotePolicy's rollout forward on its fused routes (16-bit stream, block stack in one kernel, pooled critic), enqueued natively.
//
// Composed in Python the forward was 29 ops: 0.45 ms of host time, another 0.35 for the ~60 casts and copies that follow an
// optimizer step - what one env, and a small update, then took.  Here the weights that the kernels read are one image, packed from
// the masters by three launches, and the forward is one call (or four, where the caller runs the critic on a second stream): the
// four encoders share a launch, LayerNorms read and write strided rows, so that neither the torso rows nor the value MLP's input
// is copied together.  Every kernel and its operands are those of the op-by-op forward: the same bits.
// One env, recipe shape: 419 -> 180 us, 145 with the chains of note_readout.hip, 68 of them the block stack (blocks_latency.hip: from
// 206); a captured rollout step of 2048 envs, default shape: 217 -> 180 us, 151 with the chains; the update of 1500 envs: 3.7 -> 3.3 ms.
#include "note_readout.h"
#include "note_train.h"

namespace {

constexpr int T_TOK = N_LEAD + N_NOTES, READOUT_PARTS = BSRL_NOTE_ACTOR | BSRL_NOTE_CRITIC | BSRL_NOTE_VALUE, READOUT_MOST = 32, LDS_MAX = 160 * 1024;
constexpr float MASKED_LOGIT = -1.0e9f;              // lanes past a head's gear count

bsrl_blocks_desc stack_of(const bsrl_note_desc& d) { return {d.n_blocks, d.d, d.n_heads, d.ffn, T_TOK, BSRL_ACT_RELU, N_LEAD, d.dtype}; }

struct Image {
    u16 *w0[4], *w2[4], *wp, *wf1, *wf2, *wh, *wcq, *wqk, *wvo, *wco, *m0, *m2, *m4; float* bh; void* blocks;
    ReadoutMat fr[READOUT_MATS]; int n_fr = 0; size_t bytes;              // wp .. m4 once more, as note_readout.hip streams them
    Image(const bsrl_note_desc& d, char* base) {
        Bump b{base};
        const bsrl_blocks_desc s = stack_of(d);
        const int64_t D = d.d, TR = d.trunk, H = d.hidden, HD = (int64_t)d.n_heads * D, NL = (int64_t)N_HEADS_ACT * d.n_gears;
        auto mat = [&](int64_t r, int64_t c) { return b.take<u16>((size_t)(r * c)); };
        blocks = b.take<char>((size_t)bsrl_blocks_pack_size(&s));
        for (int e = 0; e < 4; ++e) { w0[e] = mat(D, PITCH); w2[e] = mat(D, D); }
        wp = mat(TR, N_LEAD * D); wf1 = mat(H, TR); wf2 = mat(TR, H); wh = mat(NL, TR); bh = b.take<float>(NL);
        wcq = mat(D, D); wqk = mat(HD, D); wvo = mat(D, HD); wco = mat(D, D);
        m0 = mat(TR, D + TR); m2 = mat(TR, TR); m4 = mat(d.bins, TR);
        if (TR % 64 == 0 && TR <= 384 && H % 64 == 0) {
            auto frag = [&](const u16* src, int64_t r, int64_t c) { fr[n_fr++] = {src, b.take<u16>((size_t)readout_frag_elems(r, c)), (int)r, (int)c}; };
            frag(wp, TR, N_LEAD * D); frag(wf1, H, TR); frag(wf2, TR, H); frag(wh, NL, TR);
            frag(wcq, D, D); frag(wqk, HD, D); frag(wvo, D, HD); frag(wco, D, D);
            frag(m0, TR, D + TR); frag(m2, TR, TR); frag(m4, d.bins, TR);
            b.take<char>(READOUT_SLACK);
        }
        bytes = b.used;
    }
};

struct Work {
    u16 *in[4], *bias, *x, *lead, *xres, *t, *u, *r, *t2, *z, *ln, *q, *qk, *pool, *att, *c1, *c2; float* vl; int4* pairs; int* tiles; size_t bytes;
    Work(const bsrl_note_desc& d, int64_t B, char* base) {
        Bump b{base};
        const int64_t D = d.d, TR = d.trunk, HD = (int64_t)d.n_heads * D;
        auto mat = [&](int64_t r, int64_t c) { return b.take<u16>((size_t)(r * c)); };
        for (int e = 0; e < 4; ++e) in[e] = mat(B * ENC_ROWS[e], PITCH);
        bias = mat(B, T_TOK); x = mat(B * T_TOK, D); lead = mat(B, N_LEAD * D); xres = mat(B * T_TOK, D);
        t = mat(B, TR); u = mat(B, TR); r = mat(B, d.hidden); t2 = mat(B, TR); z = mat(B, D + TR);
        ln = mat(B, D); q = mat(B, D); qk = mat(B, HD); pool = mat(B, HD); att = mat(B, D); c1 = mat(B, TR); c2 = mat(B, TR);
        vl = b.take<float>((size_t)(B * d.bins));
        pairs = b.take<int4>((size_t)(bsrl_blocks_pair_chunks(B) * BLOCKS_PAIR_CHUNK));
        tiles = b.take<int>((size_t)bsrl_blocks_pair_chunks(B));
        bytes = b.used;
    }
};

// Everything behind the block stack as chains around the attention pool (note_readout.hip), for widths it covers and up to
// READOUT_MOST envs per CU: two workgroups' worth of envs each, past which weights streamed once per 16 envs cost what the
// Linears' larger tiles save (8192 envs, one call against parts on two streams: 1581 / 1577 us at the recipe's widths,
// 427 / 437 at the default's; 4096: 780 / 809, 232 / 262; 2048: 429 / 449, 143 / 175).
struct Readout {
    ReadoutArgs a = {}, v = {};
    size_t la = 0, lv = 0;
    bool ok = false;
    Readout(const bsrl_note_desc& d, const float* const* params, const Image& m, const Work& w, const float* centers, float* logits, float* value, int64_t B) {
        const int D = d.d, TR = d.trunk, H = d.hidden, HD = d.n_heads * D, NL = N_HEADS_ACT * d.n_gears;
        if (!m.n_fr || B > READOUT_MOST * (int64_t)bsrl_cus()) return;
        const NoteIndex at{d.n_blocks};
        const float* const* t = params + at.p_trunk();
        const float* const* c = params + at.p_critic();
        enum { WP, WF1, WF2, WH, WCQ, WQK, WVO, WCO, M0, M2, M4 };              // Image's order
        a.B = v.B = B;
        auto linear = [&](int W, const float* b, int in, int out, int relu = 0, int res = -1) {
            return ReadoutStep{m.fr[W].dst, b, nullptr, nullptr, 0, READOUT_LINEAR, m.fr[W].K, m.fr[W].M, in, out, res, relu, 0, 0};
        };
        auto to = [](ReadoutStep s, void* g, int64_t ld, int f32) { s.gout = g; s.gld = ld; s.f32 = f32; return s; };
        auto ln = [](const float* const* wb, int K, int in, int out) { return ReadoutStep{nullptr, wb[0], wb[1], nullptr, 0, READOUT_LN, K, 0, in, out, -1, 0, 0, 0}; };
        auto room = [](int& used, int K) { const int r = used; used += K * 2; return r; };          // K / 8 pieces of 16 envs
        int used[3] = {0, 0, 0};
        {   // actor: trunk and heads
            int& u = used[0];
            const int z = room(u, N_LEAD * D), x = room(u, TR), y = room(u, TR), h = room(u, H);
            ReadoutProg& p = a.prog[0];
            p.in[0] = {w.lead, N_LEAD * D, N_LEAD * D, z}; p.n_in = 1; p.n = 6;
            p.step[0] = linear(WP, t[1], z, x);
            p.step[1] = ln(t + 2, TR, x, y);
            p.step[2] = linear(WF1, t[5], y, h, 1);
            p.step[3] = linear(WF2, t[7], h, y, 0, x);
            p.step[4] = to(ln(t + 8, TR, y, x), w.z + D, D + TR, 0);
            p.step[5] = to(linear(WH, m.bh, x, -1), logits, NL, 1);
        }
        {   // critic: the torso token's query, folded with the keys' projection
            int& u = used[1];
            const int x = room(u, D), y = room(u, D);
            ReadoutProg& p = a.prog[1];
            p.in[0] = {w.xres + 2 * D, T_TOK * D, D, x}; p.n_in = 1; p.n = 3;
            p.step[0] = ln(c, D, x, y);
            p.step[1] = linear(WCQ, c[3], y, x);
            p.step[2] = to(linear(WQK, nullptr, x, -1), w.qk, HD, 0);
        }
        {   // value: the pooled rows' projections and the MLP
            int& u = used[2];
            const int pool = room(u, HD), x = room(u, D), z = room(u, D + TR), h1 = room(u, TR), h2 = room(u, TR), bins = room(u, (d.bins + 3) / 4 * 4 * 2);
            ReadoutProg& p = v.prog[0];
            p.in[0] = {w.pool, HD, HD, pool}; p.in[1] = {w.z + D, D + TR, TR, z + D * 2}; p.n_in = 2; p.n = 6;
            p.step[0] = linear(WVO, c[7], pool, x);
            p.step[1] = linear(WCO, c[9], x, z);
            p.step[2] = linear(M0, c[11], z, h1, 1);
            p.step[3] = linear(M2, c[13], h1, h2, 1);
            p.step[4] = linear(M4, c[15], h2, bins);
            p.step[4].f32 = 1;
            p.step[5] = {nullptr, centers, nullptr, value, 0, READOUT_EXPECT, d.bins, 0, bins, -1, -1, 0, 0};
        }
        la = bsrl_note_readout_lds(a, 2, (size_t)(used[0] > used[1] ? used[0] : used[1]) * 16);
        lv = bsrl_note_readout_lds(v, 1, (size_t)used[2] * 16);
        ok = la <= LDS_MAX && lv <= LDS_MAX;
    }
};

bool desc_ok(const bsrl_note_desc* d) {
    if (!d || (d->dtype != BSRL_F16 && d->dtype != BSRL_BF16) || (d->d != 128 && d->d != 192) || d->n_heads < 1 || d->n_heads > 16 || d->d % d->n_heads != 0 ||
        d->trunk < 8 || d->trunk % 8 != 0 || d->trunk > 2048 || d->hidden < 8 || d->hidden % 8 != 0 || d->hidden > 8192 || d->n_gears < 1 ||
        d->n_gears > 16 || d->bins < 2 || d->bins > 4096 || d->n_blocks < 1 || d->n_blocks > BSRL_MAX_LAYERS)
        return false;
    const bsrl_blocks_desc s = stack_of(*d);
    return bsrl_blocks_pack_size(&s) > 0;
}

}  // namespace

extern "C" int64_t bsrl_note_pack_size(const bsrl_note_desc* d) { return desc_ok(d) ? (int64_t)Image(*d, nullptr).bytes : 0; }
extern "C" int64_t bsrl_note_forward_size(const bsrl_note_desc* d, int64_t B) {
    return desc_ok(d) && B >= 1 && B * T_TOK <= 0x7fffffffLL ? (int64_t)Work(*d, B, nullptr).bytes : 0;
}

extern "C" int bsrl_note_one_call(const bsrl_note_desc* d, int64_t B) {
    if (!desc_ok(d) || B < 1) return 0;
    static const float* const none[16 + 16 * BSRL_MAX_LAYERS + 10 + 2 * N_HEADS_ACT + 16] = {};
    return Readout(*d, none, Image(*d, nullptr), Work(*d, B, nullptr), nullptr, nullptr, nullptr, B).ok;
}

extern "C" int bsrl_note_pairs_pay(const bsrl_note_desc* d, int64_t B, int64_t tiles) {
    if (!desc_ok(d) || B < 1 || tiles < 0) return 0;
    return blocks_pairs_pay(blocks_pair_plan(nullptr, 0, bsrl_cus(), B, d->n_blocks, d->ffn), tiles);
}

extern "C" int bsrl_note_pack(const bsrl_note_desc* d, const float* const* params, const int32_t* gears, void* image, bsrl_stream stream) {
    if (!desc_ok(d)) return BSRL_UNSUPPORTED;
    if (!params || !gears || !image || !bsrl_aligned(image, 256)) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_pack: null pointer or unaligned image");
    for (int j = 0; j < N_HEADS_ACT; ++j) if (gears[j] < 1 || gears[j] > d->n_gears) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_pack: head %d has %d gears", j, gears[j]);
    const NoteIndex at{d->n_blocks};
    const Image m(*d, static_cast<char*>(image));
    const int64_t D = d->d, TR = d->trunk, H = d->hidden, NH = d->n_heads, dh = D / NH, K = d->n_gears;
    const bsrl_blocks_desc s = stack_of(*d);
    bsrl_blocks_params bp = {};
    for (int i = 0; i < d->n_blocks; ++i) {
        const float** f = reinterpret_cast<const float**>(&bp.blk[i]);       // the pairs' order is the struct's
        for (int j = 0; j < 16; ++j) f[j] = params[at.p_blk(i) + j];
    }
    const int rc = bsrl_blocks_pack(&s, &bp, m.blocks, stream);
    if (rc != BSRL_OK) return rc;
    Packer k(static_cast<hipStream_t>(stream), d->dtype);
    for (int e = 0; e < 4; ++e) {
        k.add(params[4 * e], D, note_enc_in(*d, e), m.w0[e], PITCH, nullptr, 0, 0, PITCH);
        k.add(params[4 * e + 2], D, D, m.w2[e], D, nullptr, 0);
    }
    const float* const* p = params + at.p_trunk();
    k.add(p[0], TR, N_LEAD * D, m.wp, N_LEAD * D, nullptr, 0);
    k.add(p[4], H, TR, m.wf1, TR, nullptr, 0);
    k.add(p[6], TR, H, m.wf2, H, nullptr, 0);
    p = params + at.p_heads();
    for (int j = 0; j < N_HEADS_ACT; ++j) {
        k.add(p[2 * j], gears[j], TR, m.wh + j * K * TR, TR, nullptr, 0, K);
        k.bias(p[2 * j + 1], gears[j], m.bh + j * K, K, MASKED_LOGIT);
    }
    p = params + at.p_critic();
    k.add(p[2], D, D, m.wcq, D, nullptr, 0);
    for (int64_t h = 0; h < NH; ++h) {       // block-structured: Wk_h^T behind the query, Wv_h behind the pooled rows, zeros between (the image starts zeroed)
        k.add(p[4] + h * dh * D, dh, D, nullptr, 0, m.wqk + h * D * D + h * dh, D);
        k.add(p[6] + h * dh * D, dh, D, m.wvo + h * dh * NH * D + h * D, NH * D, nullptr, 0);
    }
    k.add(p[8], D, D, m.wco, D, nullptr, 0);
    k.add(p[10], TR, D + TR, m.m0, D + TR, nullptr, 0);
    k.add(p[12], TR, TR, m.m2, TR, nullptr, 0);
    k.add(p[14], d->bins, TR, m.m4, TR, nullptr, 0);
    k.flush();
    BSRL_CHECK_LAUNCH("bsrl_note_pack");
    return m.n_fr ? bsrl_note_readout_frags(m.fr, m.n_fr, static_cast<hipStream_t>(stream)) : BSRL_OK;
}

extern "C" int bsrl_note_forward(const bsrl_note_desc* d, const float* const* params, const void* image, const void* obs, int64_t obs_ld, int obs_dtype,
                                 const int32_t* saber_idx, const int32_t* body_idx, const float* centers, float* logits, float* value, int64_t B, int parts,
                                 void* workspace, int64_t workspace_bytes, bsrl_stream stream) {
    return bsrl_note_forward_saving(d, params, image, obs, obs_ld, obs_dtype, saber_idx, body_idx, centers, logits, value, B, parts, workspace, workspace_bytes,
                                    nullptr, 0, stream);
}

extern "C" int bsrl_note_forward_saving(const bsrl_note_desc* d, const float* const* params, const void* image, const void* obs, int64_t obs_ld, int obs_dtype,
                                        const int32_t* saber_idx, const int32_t* body_idx, const float* centers, float* logits, float* value, int64_t B,
                                        int parts, void* workspace, int64_t workspace_bytes, void* saved, int64_t saved_bytes, bsrl_stream stream) {
    if (!desc_ok(d)) return BSRL_UNSUPPORTED;
    if (!params || !image || !obs || !saber_idx || !body_idx || !centers || !logits || !value || B < 1) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_forward: bad argument");
    const int64_t need = bsrl_note_forward_size(d, B);
    if (!need || !workspace || workspace_bytes < need || !bsrl_aligned(workspace, 256) || !bsrl_aligned(image, 256))
        BSRL_FAIL(BSRL_EINVAL, "bsrl_note_forward: workspace too small or unaligned");
    const NoteIndex at{d->n_blocks};
    const Image m(*d, static_cast<char*>(const_cast<void*>(image)));
    const Work w(*d, B, static_cast<char*>(workspace));
    BlocksSave save = {};
    if (saved) {
        if (!note_train_saves(*d, B)) return BSRL_UNSUPPORTED;
        if (saved_bytes < bsrl_note_train_size(d, B, 0) || !bsrl_aligned(saved, 256)) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_forward_saving: saved too small or unaligned");
        save = note_train_blocks(*d, B, saved);
    }
    const int64_t D = d->d, TR = d->trunk, H = d->hidden, HD = (int64_t)d->n_heads * D, NL = (int64_t)N_HEADS_ACT * d->n_gears;
    const int dt = d->dtype;
    hipStream_t st = static_cast<hipStream_t>(stream);
#define STEP(call) do { const int rc_ = (call); if (rc_ != BSRL_OK) return rc_; } while (0)
    auto linear = [&](const void* x, int64_t ldx, const void* W, const float* b, void* y, int64_t ldy, int64_t K, int64_t M, int act = BSRL_ACT_NONE,
                      const void* res = nullptr, bool f32 = false) {
        const LinArgs a{x, ldx, W, b, res, M, y, ldy, nullptr, 0, 0, B, (int)K, (int)M, f32, 0, 0, nullptr, 0};
        return bsrl_linear_run(a, act, dt, f32 ? BSRL_F32 : dt, st, "bsrl_note_forward");
    };
    auto ln = [&](const void* x, int64_t ldx, const float* const* wb, void* y, int64_t ldy, int64_t dim) {
        return bsrl_ln_rows(x, ldx, wb[0], wb[1], y, ldy, nullptr, nullptr, B, nullptr, B, dim, 1e-5f, dt, stream);
    };
    if (parts & BSRL_NOTE_STACK) {
        STEP(bsrl_note_frontend_padded(obs, obs_ld, obs_dtype, saber_idx, body_idx, (d->note_geo ? BSRL_NOTE_GEO : 0) | BSRL_NOTE_ZERO_MASKED, d->flux, d->z_asinh,
                                       w.in[0], w.in[1], w.in[2], w.in[3], w.bias, B, dt, stream));
        Mlp2Args e4[4];
        for (int e = 0; e < 4; ++e) {
            const LinArgs l2{nullptr, 0, m.w2[e], params[4 * e + 3], nullptr, 0, w.x + ENC_AT[e] * D, D, nullptr, 0, 0, B * ENC_ROWS[e], (int)D, (int)D, 0,
                             ENC_ROWS[e], T_TOK * D, nullptr, 0};
            e4[e] = {l2, w.in[e], PITCH, m.w0[e], params[4 * e + 1]};
        }
        if (!bsrl_mlp2_stream(e4, 4, PITCH, dt, st)) return BSRL_UNSUPPORTED;
        const bsrl_blocks_desc s = stack_of(*d);
        const int64_t frags = bsrl_blocks_pack_size(&s) - (int64_t)s.n_layers * (9 * D + s.ffn) * 4;
        const BlocksPairPlan plan = blocks_pair_plan(w.tiles, (int)bsrl_blocks_pair_chunks(B), bsrl_cus(), B, s.n_layers, s.ffn);
        const BlocksPairArgs p{static_cast<const uint4*>(m.blocks), reinterpret_cast<const float*>(static_cast<const char*>(m.blocks) + frags), w.x, w.bias, w.xres,
                               w.lead, w.pairs, plan, s.n_layers, s.ffn, T_TOK, N_LEAD, (int)(frags / (D / 16 * 1024))};
        if (saved) STEP(bsrl_blocks_pair_save(p, save, dt, st));
        else {
            const int rc = bsrl_blocks_pair(p, d->d, dt, st);
            if (rc != BSRL_UNSUPPORTED) STEP(rc);
            STEP(bsrl_blocks_unless(&s, m.blocks, w.x, w.bias, w.xres, w.lead, B, rc == BSRL_OK ? &plan : nullptr, stream));
        }
    }
    if ((parts & READOUT_PARTS) == READOUT_PARTS) {
        const Readout r(*d, params, m, w, centers, logits, value, B);
        if (r.ok) {
            const float* const* c = params + at.p_critic();
            STEP(bsrl_note_readout(r.a, 2, r.la, dt, st));
            STEP(bsrl_critic_pool(w.xres, c[0], c[1], 1e-5f, w.qk, w.bias, w.pool, B, T_TOK, D, d->n_heads, dt, stream));
            return bsrl_note_readout(r.v, 1, r.lv, dt, st);
        }
    }
    if (parts & BSRL_NOTE_ACTOR) {
        const float* const* p = params + at.p_trunk();
        STEP(linear(w.lead, N_LEAD * D, m.wp, p[1], w.t, TR, N_LEAD * D, TR));
        STEP(ln(w.t, TR, p + 2, w.u, TR, TR));
        STEP(linear(w.u, TR, m.wf1, p[5], w.r, H, TR, H, BSRL_ACT_RELU));
        STEP(linear(w.r, H, m.wf2, p[7], w.t2, TR, H, TR, BSRL_ACT_NONE, w.t));
        STEP(ln(w.t2, TR, p + 8, w.z + D, D + TR, TR));                      // beside the critic's attention output
        STEP(linear(w.z + D, D + TR, m.wh, m.bh, logits, NL, TR, NL, BSRL_ACT_NONE, nullptr, true));
    }
    const float* const* p = params + at.p_critic();
    if (parts & BSRL_NOTE_CRITIC) {
        STEP(ln(w.xres + 2 * D, T_TOK * D, p, w.ln, D, D));                  // the torso token's rows
        STEP(linear(w.ln, D, m.wcq, p[3], w.q, D, D, D));
        STEP(linear(w.q, D, m.wqk, nullptr, w.qk, HD, D, HD));               // Wk_h^T q_h per head
        STEP(bsrl_critic_pool(w.xres, p[0], p[1], 1e-5f, w.qk, w.bias, w.pool, B, T_TOK, D, d->n_heads, dt, stream));
        STEP(linear(w.pool, HD, m.wvo, p[7], w.att, D, HD, D));              // Wv_h pooled_h + bv_h
        STEP(linear(w.att, D, m.wco, p[9], w.z, D + TR, D, D));
    }
    if (parts & BSRL_NOTE_VALUE) {
        STEP(linear(w.z, D + TR, m.m0, p[11], w.c1, TR, D + TR, TR, BSRL_ACT_RELU));
        STEP(linear(w.c1, TR, m.m2, p[13], w.c2, TR, TR, TR, BSRL_ACT_RELU));
        STEP(linear(w.c2, TR, m.m4, p[15], w.vl, d->bins, TR, d->bins, BSRL_ACT_NONE, nullptr, true));
        STEP(bsrl_softmax_expect(w.vl, centers, value, B, d->bins, stream));
    }
#undef STEP
    return BSRL_OK;
}
