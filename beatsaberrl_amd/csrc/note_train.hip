// NotePolicy's update on the 16-bit stream, forward and backward, each enqueued by one call over the compacted token stream.
//
// Composed in Python (one autograd Function per op over the full 29-token stream) an update was 427 launches at three blocks and
// the host was the bound: 6.1 ms of Python for 3.2 ms of kernels at 1500 envs; at 16384 envs the kernels were, and a third of
// their rows were notes that are not there.  Here
//   * the stream holds the 5 lead tokens of every env and the notes that attention can see (ragged.hip): a note that is masked
//     has weight zero in every softmax, so neither an output nor a gradient depends on its row.  The row count stays on the device.
//     Attention keeps its keys in their slots of the full stream: the forward's bits are the op-by-op update's;
//   * the masters become the forward's weights and the backward's transposed ones in one pass (pack_kernel);
//   * gradients that torch would add up in passes of their own ride in epilogues: residual branches in ln_bwd (gx) and in the
//     data-gradient GEMMs (res = y on the lead rows);
//   * every launch is enqueued here, ~3 us of host time each.
// Past a round of the rollout's paired block stack (blocks_pair.hip, d = 192, more than 8 envs per CU) the stack's launch leaves the blocks'
// activations here and this forward is what lies in front of it and behind it: 17.6 -> 14.2 ms for 16384 envs at the recipe's shape.  Up to
// there the bin logits keep the op-by-op update's bits; past it the forward is the rollout's, whose stream is not rounded between blocks (its
// error against 64 bits: blocks_pair.hip).  An env's bin logits and gradients differ by such roundings between the two.
// Update of 16384 envs, recipe shape, before that: 26.1 -> 19.6 ms; 1500 envs, default shape: 6.4 -> 3.7 ms (the rollout's forward, the loss
// and torch's part of the backward included).
#include "note_train.h"

namespace {

// dst (rows, pad) 16-bit = src (rows, n) fp32, zero past n
template <typename DT>
__global__ __launch_bounds__(256) void narrow_kernel(const float* __restrict__ src, int n, u16* __restrict__ dst, int pad, int64_t total) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t row = i / pad;
    const int c = (int)(i - row * pad);
    dst[i] = c < n ? DT::from_f(src[row * n + c]) : (u16)0;
}

// rows of 16-byte pieces: dst row r from src row (r / group) gstride + (r % group) sld (strides in pieces)
__global__ __launch_bounds__(256) void rows_copy_kernel(uint4* __restrict__ dst, int64_t dld, const uint4* __restrict__ src, int64_t sld,
                                                        int group, int64_t gstride, int64_t rows, int pieces) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= rows * pieces) return;
    const int64_t r = i / pieces;
    const int p = (int)(i - r * pieces);
    dst[r * dld + p] = src[(r / group) * gstride + (r % group) * sld + p];
}

struct Stats { float *mean, *rstd; };

// ---- what the forward leaves for the backward ----------------------------------------------------------------------------
struct Saved {
    struct Enc { u16 *in, *hid, *w0, *w2, *t2; } enc[4];
    struct Blk { u16 *x, *h, *qkv, *q, *att, *xm, *h2, *hid; Stats s1, s2; u16 *wqkv, *tqkv, *tq, *wo, *to, *w0, *t0, *w2, *t2; float* bqkv; } blk[BSRL_MAX_LAYERS];
    int32_t *noff, *cnt; u16* bias; uint8_t* slots; float* apart;               // apart: 1 where the blocks' q, k, v lie head after head (blocks_pair.h), else 0
    u16 *lead, *t, *u, *r, *t2; Stats s1, s2;                                  // trunk
    u16 *wp, *tp, *wf1, *tf1, *wf2, *tf2, *th;
    u16 *hv, *cq, *ckv, *catt, *z, *c1, *c2; Stats sc;                              // critic
    u16 *wcq, *tcq, *wckv, *tckv, *wco, *tco, *m0, *tm0, *m2, *tm2, *m4, *tm4; float* bckv;
    size_t bytes;
};

struct Net : NoteIndex {
    const bsrl_note_desc& d; int64_t B, R, D, F, TR, H, NL, BINS;
    explicit Net(const bsrl_note_desc& d_, int64_t B_) : NoteIndex{d_.n_blocks}, d(d_), B(B_), R(B_ * (N_LEAD + N_NOTES)), D(d_.d), F(d_.ffn), TR(d_.trunk),
                                                         H(d_.hidden), NL((int64_t)N_HEADS_ACT * d_.n_gears), BINS(d_.bins) {}
    int64_t enc_in(int e) const { return note_enc_in(d, e); }

    Saved saved(char* base) const {
        Saved s; Bump b{base};
        auto mat = [&](int64_t r, int64_t c) { return b.take<u16>((size_t)(r * c)); };
        auto stats = [&](int64_t r) { Stats st; st.mean = b.take<float>(r); st.rstd = b.take<float>(r); return st; };
        s.noff = b.take<int32_t>(B + 1); s.cnt = b.take<int32_t>(B); s.bias = b.take<u16>(B * N_NOTES); s.slots = b.take<uint8_t>(B * 32); s.apart = b.take<float>(1);
        for (int e = 0; e < 4; ++e) s.enc[e] = {mat(B * ENC_ROWS[e], PITCH), mat(B * ENC_ROWS[e], D), mat(D, PITCH), mat(D, D), mat(D, D)};
        for (int i = 0; i < L; ++i) {
            auto& k = s.blk[i];
            const bool last = i + 1 == L;
            const int64_t rows = last ? N_LEAD * B : R;                             // the final block's rows behind its keys and values
            k.x = mat(R, D); k.h = mat(R, D); k.qkv = mat(R, last ? 2 * D : 3 * D); k.q = last ? mat(rows, D) : k.qkv;
            k.att = mat(rows, D); k.xm = mat(rows, D); k.h2 = mat(rows, D); k.hid = mat(rows, F);
            k.s1 = stats(R); k.s2 = stats(rows);
            k.wqkv = mat(3 * D, D); k.tqkv = mat(D, last ? 2 * D : 3 * D); k.tq = last ? mat(D, D) : nullptr;
            k.wo = mat(D, D); k.to = mat(D, D); k.w0 = mat(F, D); k.t0 = mat(D, F); k.w2 = mat(D, F); k.t2 = mat(F, D);
            k.bqkv = b.take<float>(3 * D);
        }
        s.lead = mat(B, N_LEAD * D); s.t = mat(B, TR); s.u = mat(B, TR); s.r = mat(B, H); s.t2 = mat(B, TR);
        s.s1 = stats(B); s.s2 = stats(B);
        s.wp = mat(TR, N_LEAD * D); s.tp = mat(N_LEAD * D, TR); s.wf1 = mat(H, TR); s.tf1 = mat(TR, H); s.wf2 = mat(TR, H); s.tf2 = mat(H, TR);
        s.th = mat(TR, pad32(NL));
        s.hv = mat(R, D); s.sc = stats(R); s.cq = mat(B, D); s.ckv = mat(R, 2 * D); s.catt = mat(B, D); s.z = mat(B, D + TR); s.c1 = mat(B, TR); s.c2 = mat(B, TR);
        s.wcq = mat(D, D); s.tcq = mat(D, D); s.wckv = mat(2 * D, D); s.tckv = mat(D, 2 * D); s.wco = mat(D, D); s.tco = mat(D, D);
        s.m0 = mat(TR, D + TR); s.tm0 = mat(D + TR, TR); s.m2 = mat(TR, TR); s.tm2 = mat(TR, TR); s.m4 = mat(pad32(BINS), TR); s.tm4 = mat(TR, pad32(BINS));
        s.bckv = b.take<float>(2 * D);
        s.bytes = b.used;
        return s;
    }

    // offset of every parameter's gradient in the flat fp32 buffer, and its length: q | k | v (k | v of the critic) and the
    // heads lie together, weights then biases, as their packed projections' weight gradients are written
    int64_t layout(int64_t* off) const {
        int64_t at = 0;
        auto put = [&](int p, int64_t n) { off[p] = at; at += n; };
        auto align = [&] { at = (at + 63) / 64 * 64; };
        auto lin = [&](int p, int64_t m, int64_t k) { put(p, m * k); align(); put(p + 1, m); align(); };
        auto ln = [&](int p, int64_t n) { put(p, n); align(); put(p + 1, n); align(); };
        for (int e = 0; e < 4; ++e) { lin(4 * e, D, enc_in(e)); lin(4 * e + 2, D, D); }
        for (int i = 0; i < L; ++i) {
            const int p = p_blk(i);
            ln(p, D);
            for (int j = 0; j < 3; ++j) put(p + 2 + 2 * j, D * D);
            align();
            for (int j = 0; j < 3; ++j) put(p + 3 + 2 * j, D);
            align();
            lin(p + 8, D, D); ln(p + 10, D); lin(p + 12, F, D); lin(p + 14, D, F);
        }
        int p = p_trunk();
        lin(p, TR, N_LEAD * D); ln(p + 2, TR); lin(p + 4, H, TR); lin(p + 6, TR, H); ln(p + 8, TR);
        p = p_heads();
        for (int j = 0; j < N_HEADS_ACT; ++j) put(p + 2 * j, d.n_gears * TR);
        align();
        for (int j = 0; j < N_HEADS_ACT; ++j) put(p + 2 * j + 1, d.n_gears);
        align();
        p = p_critic();
        ln(p, D); lin(p + 2, D, D);
        put(p + 4, D * D); put(p + 6, D * D); align(); put(p + 5, D); put(p + 7, D); align();
        lin(p + 8, D, D); lin(p + 10, TR, D + TR); lin(p + 12, TR, TR); lin(p + 14, BINS, TR);
        return at;
    }
};

struct Scratch {
    u16 *dl, *dv, *dc2, *dc1, *dz, *dhf, *dr, *drh, *du, *dt, *g5, *gm, *dm, *xm, *dqkv, *g, *gx, *dcat, *dcq, *dq5, *es, *el, *eh[4];
    void *ws_wg, *ws_ln; int64_t wg_bytes; size_t bytes;
    Scratch(const Net& n, char* base) {
        Bump b{base};
        auto mat = [&](int64_t r, int64_t c) { return b.take<u16>((size_t)(r * c)); };
        const int64_t B = n.B, R = n.R, D = n.D, F = n.F, TR = n.TR, H = n.H;
        dl = mat(B, pad32(n.NL)); dv = mat(B, pad32(n.BINS)); dc2 = mat(B, TR); dc1 = mat(B, TR); dz = mat(B, D + TR);
        dhf = mat(B, TR); dr = mat(B, TR); drh = mat(B, H); du = mat(B, TR); dt = mat(B, TR); g5 = mat(B, N_LEAD * D);
        gm = mat(n.L > 1 ? R : N_LEAD * B, F); dm = mat(R, D); xm = mat(R, D); dqkv = mat(R, 3 * D); g = mat(R, D); gx = mat(R, D);
        dcat = mat(B, D); dcq = mat(B, D); dq5 = mat(N_LEAD * B, D); es = mat(2 * B, D); el = mat(2 * B, D);
        for (int e = 0; e < 4; ++e) eh[e] = mat(B * ENC_ROWS[e], D);
        // the weight gradients come in four batches: heads (trunk, critic), final block, other blocks, encoders
        struct Shape { int64_t rows, M, K, MO; };
        const int64_t LB = N_LEAD * B, BP = pad32(n.BINS), HP = pad32(n.NL);
        const std::initializer_list<Shape> batches[] = {
            {{B, BP, TR, n.BINS}, {B, TR, TR, TR}, {B, TR, D + TR, TR}, {B, D, D, D}, {R, 2 * D, D, 2 * D}, {B, D, D, D}, {B, HP, TR, n.NL}, {B, TR, H, TR},
             {B, H, TR, H}, {B, TR, N_LEAD * D, TR}},
            {{LB, D, F, D}, {LB, F, D, F}, {LB, D, D, D}, {R, 2 * D, D, 2 * D}, {LB, D, D, D}},
            {{R, D, F, D}, {R, F, D, F}, {R, D, D, D}, {R, 3 * D, D, 3 * D}},
            {{2 * B, D, D, D}, {2 * B, D, PITCH, D}, {B, D, D, D}, {B, D, PITCH, D}, {2 * B, D, D, D}, {2 * B, D, PITCH, D}, {N_NOTES * B, D, D, D},
             {N_NOTES * B, D, PITCH, D}}};
        wg_bytes = 0;
        for (const auto& batch : batches) {
            WgradProblem p[12];
            int k = 0;
            for (const Shape& q : batch) p[k++] = {nullptr, q.M, nullptr, q.K, nullptr, nullptr, q.rows, nullptr, 0, q.M, q.K, q.MO, q.K};
            const int64_t w = bsrl_wgrad_batch_size(p, k);
            if (w > wg_bytes) wg_bytes = w;
        }
        ws_wg = b.take<char>(wg_bytes);
        const int64_t l0 = bsrl_ln_bwd_workspace_size(D), l1 = bsrl_ln_bwd_workspace_size(TR);
        ws_ln = b.take<char>(l0 > l1 ? l0 : l1);
        bytes = b.used;
    }
};

bool desc_ok(const bsrl_note_desc* d) {
    return d && (d->dtype == BSRL_F16 || d->dtype == BSRL_BF16) && d->n_blocks >= 1 && d->n_blocks <= BSRL_MAX_LAYERS && d->n_heads >= 1 &&
           d->d >= 32 && d->d % 32 == 0 && d->d % d->n_heads == 0 && d->d <= 2048 && d->ffn >= 32 && d->ffn % 32 == 0 && d->ffn <= 8192 &&
           d->trunk >= 32 && d->trunk % 32 == 0 && d->trunk <= 2048 && d->hidden >= 32 && d->hidden % 32 == 0 && d->hidden <= 8192 &&
           d->n_gears >= 1 && d->n_gears <= 16 && d->bins >= 2 && d->bins <= 4096 &&
           bsrl_attn_bwd_ragged_ok(N_LEAD + N_NOTES, d->n_heads, d->d / d->n_heads, d->dtype);
}

void pack_all(const Net& n, const Saved& s, const float* const* P, bool apart, hipStream_t st) {
    Packer k(st, n.d.dtype);
    k.add(P[0], 1, 0, s.apart, 1, nullptr, 0, 1, 1, true, apart ? 1.f : 0.f);      // (nothing but its fill)
    const int64_t D = n.D, F = n.F, TR = n.TR, H = n.H;
    for (int e = 0; e < 4; ++e) {
        k.add(P[4 * e], D, n.enc_in(e), s.enc[e].w0, PITCH, nullptr, 0, 0, PITCH);
        k.add(P[4 * e + 2], D, D, s.enc[e].w2, D, s.enc[e].t2, D);
    }
    for (int i = 0; i < n.L; ++i) {
        const auto& b = s.blk[i];
        const float* const* p = P + n.p_blk(i);
        const bool last = i + 1 == n.L;
        for (int j = 0; j < 3; ++j) {
            u16* t = !last ? b.tqkv + j * D : j == 0 ? b.tq : b.tqkv + (j - 1) * D;
            k.add(p[2 + 2 * j], D, D, b.wqkv + j * D * D, D, t, !last ? 3 * D : j == 0 ? D : 2 * D);
            k.bias(p[3 + 2 * j], D, b.bqkv + j * D);
        }
        k.add(p[8], D, D, b.wo, D, b.to, D);
        k.add(p[12], F, D, b.w0, D, b.t0, F);
        k.add(p[14], D, F, b.w2, F, b.t2, D);
    }
    const float* const* p = P + n.p_trunk();
    k.add(p[0], TR, N_LEAD * D, s.wp, N_LEAD * D, s.tp, TR);
    k.add(p[4], H, TR, s.wf1, TR, s.tf1, H);
    k.add(p[6], TR, H, s.wf2, H, s.tf2, TR);
    p = P + n.p_heads();
    const int64_t HP = pad32(n.NL), g = n.d.n_gears;
    for (int j = 0; j < N_HEADS_ACT; ++j)
        k.add(p[2 * j], g, TR, nullptr, 0, s.th + j * g, HP, j + 1 == N_HEADS_ACT ? g + HP - n.NL : g);
    p = P + n.p_critic();
    k.add(p[2], D, D, s.wcq, D, s.tcq, D);
    for (int j = 0; j < 2; ++j) {
        k.add(p[4 + 2 * j], D, D, s.wckv + j * D * D, D, s.tckv + j * D, 2 * D);
        k.bias(p[5 + 2 * j], D, s.bckv + j * D);
    }
    k.add(p[8], D, D, s.wco, D, s.tco, D);
    k.add(p[10], TR, D + TR, s.m0, D + TR, s.tm0, TR);
    k.add(p[12], TR, TR, s.m2, TR, s.tm2, TR);
    k.add(p[14], n.BINS, TR, s.m4, TR, s.tm4, pad32(n.BINS), pad32(n.BINS));
    k.flush();
}

// The ops, over all rows of the stream (`all`) or a host-side count
struct Ops {
    const Net& n; const int32_t* extra; hipStream_t st; int dt;
    // y = act(x W^T + b) (+ res); gate: the ReLU mask of a data gradient
    int linear(const void* x, int64_t ldx, const void* w, const float* b, void* y, int64_t ldy, int64_t K, int64_t M, bool all, int64_t rows,
               int act = BSRL_ACT_NONE, const void* res = nullptr, int64_t ldr = 0, const void* gate = nullptr, int64_t ldg = 0, bool f32 = false,
               int group = 0, int64_t gstride = 0) const {
        LinArgs a{x, ldx, w, b, res, ldr, y, ldy, nullptr, 0, 0, all ? n.R : rows, (int)K, (int)M, f32, group, gstride, gate, ldg};
        if (all) { a.extra = extra; a.base = N_LEAD * n.B; }
        return bsrl_linear_run(a, act, dt, f32 ? BSRL_F32 : dt, st, "bsrl_note_train");
    }
    int ln(const void* x, const float* const* wb, void* y, const Stats& s, int64_t d, bool all, int64_t rows, int64_t ldy = 0) const {
        return bsrl_ln_rows(x, d, wb[0], wb[1], y, ldy ? ldy : d, s.mean, s.rstd, all ? N_LEAD * n.B : rows, all ? extra : nullptr, all ? n.R : rows, d, 1e-5f, dt, st);
    }
    int ln_bwd(const Scratch& c, const void* x, const void* dy, const float* w, const Stats& s, const void* gx, int64_t gx_rows, void* dx, float* dw,
               float* db, int64_t d, bool all, int64_t rows) const {
        return bsrl_ln_bwd_rows(x, dy, w, s.mean, s.rstd, gx, gx_rows, dx, dw, db, nullptr, c.ws_ln, all ? N_LEAD * n.B : rows, all ? extra : nullptr,
                                all ? n.R : rows, d, dt, st);
    }
    WgradProblem wgrad(const void* dy, int64_t lddy, const void* x, int64_t ldx, float* dw, float* db, int64_t M, int64_t K, bool all, int64_t rows,
                       int64_t MO = 0) const {
        return {dy, lddy, x, ldx, dw, db, all ? n.R : rows, all ? extra : nullptr, N_LEAD * n.B, M, K, MO ? MO : M, K};
    }
    int attn(const u16* q, int64_t q_ld, const u16* k, const u16* v, int64_t kv_ld, const Saved& s, u16* out, int64_t nq) const {
        return bsrl_attn_ragged_slots(q, q_ld, k, kv_ld, v, kv_ld, s.noff, s.slots, s.bias, out, n.D, n.B, N_LEAD, N_NOTES, nq, n.d.n_heads, n.D / n.d.n_heads, dt, st);
    }
    int attn_bwd(const u16* q, int64_t q_ld, const u16* k, const u16* v, int64_t kv_ld, const Saved& s, const u16* dout, u16* dq, u16* dk, u16* dv,
                 int64_t nq, const AttnHeadsApart* apart = nullptr) const {
        return bsrl_attn_bwd_ragged(q, q_ld, k, kv_ld, v, kv_ld, s.noff, s.bias, dout, n.D, dq, q_ld, dk, kv_ld, dv, kv_ld, n.B, N_LEAD, N_NOTES, nq,
                                    n.d.n_heads, n.D / n.d.n_heads, dt, st, apart);
    }
    void copy(u16* dst, int64_t dld, const u16* src, int64_t sld, int group, int64_t gstride, int64_t rows, int64_t cols) const {
        const int64_t total = rows * (cols / 8);
        hipLaunchKernelGGL(rows_copy_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, reinterpret_cast<uint4*>(dst), dld / 8,
                           reinterpret_cast<const uint4*>(src), sld / 8, group, gstride / 8, rows, (int)(cols / 8));
    }
    void narrow(const float* src, int64_t cols, u16* dst, int64_t pad) const {
        const int64_t total = n.B * pad;
        const dim3 grid((unsigned)((total + 255) / 256));
        if (dt == BSRL_F16) hipLaunchKernelGGL(narrow_kernel<F16>, grid, dim3(256), 0, st, src, (int)cols, dst, (int)pad, total);
        else hipLaunchKernelGGL(narrow_kernel<BF16>, grid, dim3(256), 0, st, src, (int)cols, dst, (int)pad, total);
    }
};

#define STEP(call) do { const int rc_ = (call); if (rc_ != BSRL_OK) return rc_; } while (0)

// weights, offsets and the encoders; tokens: down to the first block's input, for `blocks` (else to the encoders' hidden, for the rollout's stack)
int front(const Net& n, const Saved& s, const float* const* P, const void* obs, int64_t obs_ld, int obs_dtype, const int32_t* saber_idx,
          const int32_t* body_idx, bool tokens, hipStream_t st) {
    const int64_t B = n.B, D = n.D, LB = N_LEAD * B;
    const int dt = n.d.dtype;
    pack_all(n, s, P, !tokens, st);
    STEP(bsrl_note_counts(obs, obs_ld, obs_dtype, s.cnt, B, dt, st));
    STEP(bsrl_token_offsets(s.cnt, B, N_NOTES, s.noff, st));
    STEP(bsrl_note_frontend_rows(obs, obs_ld, obs_dtype, saber_idx, body_idx, n.d.note_geo, n.d.flux, n.d.z_asinh, s.noff, s.enc[0].in, s.enc[1].in,
                                 s.enc[2].in, s.enc[3].in, s.bias, s.slots, B, dt, st));
    // tokens: the encoders write their rows of the stream
    u16* x0 = s.blk[0].x;
    for (int e = 0; e < 4; ++e) {
        const auto& k = s.enc[e];
        const float* const* p = P + 4 * e;
        LinArgs a{k.in, PITCH, k.w0, p[1], nullptr, 0, k.hid, D, nullptr, 0, 0, B * ENC_ROWS[e], PITCH, (int)D, 0, 0, 0, nullptr, 0};
        LinArgs c{k.hid, D, k.w2, p[3], nullptr, 0, x0 + ENC_AT[e] * D, D, nullptr, 0, 0, B * ENC_ROWS[e], (int)D, (int)D, 0, ENC_ROWS[e], N_LEAD * D, nullptr, 0};
        if (e == 3) { a.extra = c.extra = s.noff + B; c.y = x0 + LB * D; c.y_group = 0; c.y_gstride = 0; }
        STEP(bsrl_linear_run(a, BSRL_ACT_RELU, dt, dt, st, "bsrl_note_train"));
        if (tokens) STEP(bsrl_linear_run(c, BSRL_ACT_NONE, dt, dt, st, "bsrl_note_train"));
    }
    return BSRL_OK;
}

int blocks(const Net& n, const Saved& s, const float* const* P, hipStream_t st) {
    const int64_t B = n.B, D = n.D, F = n.F, LB = N_LEAD * B;
    const Ops o{n, s.noff + B, st, n.d.dtype};
    for (int i = 0; i < n.L; ++i) {
        const auto& k = s.blk[i];
        const float* const* p = P + n.p_blk(i);
        const bool last = i + 1 == n.L;
        STEP(o.ln(k.x, p, k.h, k.s1, D, true, 0));
        if (last) {
            STEP(o.linear(k.h, D, k.wqkv + D * D, k.bqkv + D, k.qkv, 2 * D, D, 2 * D, true, 0));
            STEP(o.linear(k.h, D, k.wqkv, k.bqkv, k.q, D, D, D, false, LB));
            STEP(o.attn(k.q, D, k.qkv, k.qkv + D, 2 * D, s, k.att, N_LEAD));
        } else {
            STEP(o.linear(k.h, D, k.wqkv, k.bqkv, k.qkv, 3 * D, D, 3 * D, true, 0));
            STEP(o.attn(k.qkv, 3 * D, k.qkv + D, k.qkv + 2 * D, 3 * D, s, k.att, 0));
        }
        STEP(o.linear(k.att, D, k.wo, p[9], k.xm, D, D, D, !last, LB, BSRL_ACT_NONE, k.x, D));
        STEP(o.ln(k.xm, p + 10, k.h2, k.s2, D, !last, LB));
        STEP(o.linear(k.h2, D, k.w0, p[13], k.hid, F, D, F, !last, LB, BSRL_ACT_RELU));
        STEP(o.linear(k.hid, F, k.w2, p[15], last ? s.lead : s.blk[i + 1].x, D, F, D, !last, LB, BSRL_ACT_NONE, k.xm, D));
    }
    return BSRL_OK;
}

// trunk and critic, from the block stack's rows
int readout(const Net& n, const Saved& s, const float* const* P, float* vlogits, hipStream_t st) {
    const int64_t B = n.B, D = n.D, TR = n.TR, H = n.H;
    const Ops o{n, s.noff + B, st, n.d.dtype};
    const float* const* p = P + n.p_trunk();
    STEP(o.linear(s.lead, N_LEAD * D, s.wp, p[1], s.t, TR, N_LEAD * D, TR, false, B));
    STEP(o.ln(s.t, p + 2, s.u, s.s1, TR, false, B));
    STEP(o.linear(s.u, TR, s.wf1, p[5], s.r, H, TR, H, false, B, BSRL_ACT_RELU));
    STEP(o.linear(s.r, H, s.wf2, p[7], s.t2, TR, H, TR, false, B, BSRL_ACT_NONE, s.t, TR));
    STEP(o.ln(s.t2, p + 8, s.z + D, s.s2, TR, false, B, D + TR));       // beside the critic's attention output: the value MLP's input
    // critic: one query per env, from its torso token
    const u16* xr = s.blk[n.L - 1].x;
    p = P + n.p_critic();
    STEP(o.ln(xr, p, s.hv, s.sc, D, true, 0));
    STEP(o.linear(s.hv + 2 * D, N_LEAD * D, s.wcq, p[3], s.cq, D, D, D, false, B));
    STEP(o.linear(s.hv, D, s.wckv, s.bckv, s.ckv, 2 * D, D, 2 * D, true, 0));
    STEP(o.attn(s.cq, D, s.ckv, s.ckv + D, 2 * D, s, s.catt, 1));
    STEP(o.linear(s.catt, D, s.wco, p[9], s.z, D + TR, D, D, false, B));
    STEP(o.linear(s.z, D + TR, s.m0, p[11], s.c1, TR, D + TR, TR, false, B, BSRL_ACT_RELU));
    STEP(o.linear(s.c1, TR, s.m2, p[13], s.c2, TR, TR, TR, false, B, BSRL_ACT_RELU));
    STEP(o.linear(s.c2, TR, s.m4, p[15], vlogits, n.BINS, TR, n.BINS, false, B, BSRL_ACT_NONE, nullptr, 0, nullptr, 0, true));
    return BSRL_OK;
}

int backward(const Net& n, const Saved& s, const Scratch& c, const float* const* P, const float* dlogits, const float* dvlogits, float* grads,
             const int64_t* off, hipStream_t st) {
    const int64_t B = n.B, D = n.D, F = n.F, TR = n.TR, H = n.H, LB = N_LEAD * B, HP = pad32(n.NL), BP = pad32(n.BINS);
    const Ops o{n, s.noff + B, st, n.d.dtype};
    auto G = [&](int p) { return grads + off[p]; };
    const auto& last = s.blk[n.L - 1];
    const bool either = note_train_saves(n.d, B);      // the forward may have been either: Saved::apart says which
    // weight gradients wait for each other: one launch per part of the net and tile shape, before their operands' buffers are used again
    WgradProblem batch[12];
    int nb = 0;
    auto flush = [&] { const int k = nb; nb = 0; return bsrl_wgrad_batch(batch, k, c.ws_wg, c.wg_bytes, n.d.dtype, st); };
    // the gradients enter the stream dtype
    o.narrow(dlogits, n.NL, c.dl, HP);
    o.narrow(dvlogits, n.BINS, c.dv, BP);
    // critic MLP and attention, down to the normalised stream (c.gx)
    int q = n.p_critic();
    batch[nb++] = o.wgrad(c.dv, BP, s.c2, TR, G(q + 14), G(q + 15), BP, TR, false, B, n.BINS);
    STEP(o.linear(c.dv, BP, s.tm4, nullptr, c.dc2, TR, BP, TR, false, B, BSRL_ACT_NONE, nullptr, 0, s.c2, TR));
    batch[nb++] = o.wgrad(c.dc2, TR, s.c1, TR, G(q + 12), G(q + 13), TR, TR, false, B);
    STEP(o.linear(c.dc2, TR, s.tm2, nullptr, c.dc1, TR, TR, TR, false, B, BSRL_ACT_NONE, nullptr, 0, s.c1, TR));
    batch[nb++] = o.wgrad(c.dc1, TR, s.z, D + TR, G(q + 10), G(q + 11), TR, D + TR, false, B);
    STEP(o.linear(c.dc1, TR, s.tm0, nullptr, c.dz, D + TR, TR, D + TR, false, B));
    batch[nb++] = o.wgrad(c.dz, D + TR, s.catt, D, G(q + 8), G(q + 9), D, D, false, B);
    STEP(o.linear(c.dz, D + TR, s.tco, nullptr, c.dcat, D, D, D, false, B));
    STEP(o.attn_bwd(s.cq, D, s.ckv, s.ckv + D, 2 * D, s, c.dcat, c.dcq, c.dqkv, c.dqkv + D, 1));
    batch[nb++] = o.wgrad(c.dqkv, 2 * D, s.hv, D, G(q + 4), G(q + 5), 2 * D, D, true, 0);
    batch[nb++] = o.wgrad(c.dcq, D, s.hv + 2 * D, N_LEAD * D, G(q + 2), G(q + 3), D, D, false, B);
    STEP(o.linear(c.dqkv, 2 * D, s.tckv, nullptr, c.gx, D, 2 * D, D, true, 0));
    STEP(o.linear(c.dcq, D, s.tcq, nullptr, c.gx + 2 * D, N_LEAD * D, D, D, false, B, BSRL_ACT_NONE, c.gx + 2 * D, N_LEAD * D));
    // heads and trunk
    q = n.p_heads();
    batch[nb++] = o.wgrad(c.dl, HP, s.z + D, D + TR, G(q), G(q + 1), HP, TR, false, B, n.NL);
    STEP(o.linear(c.dl, HP, s.th, nullptr, c.dhf, TR, HP, TR, false, B, BSRL_ACT_NONE, c.dz + D, D + TR));
    q = n.p_trunk();
    STEP(o.ln_bwd(c, s.t2, c.dhf, P[q + 8], s.s2, nullptr, 0, c.dr, G(q + 8), G(q + 9), TR, false, B));
    batch[nb++] = o.wgrad(c.dr, TR, s.r, H, G(q + 6), G(q + 7), TR, H, false, B);
    STEP(o.linear(c.dr, TR, s.tf2, nullptr, c.drh, H, TR, H, false, B, BSRL_ACT_NONE, nullptr, 0, s.r, H));
    batch[nb++] = o.wgrad(c.drh, H, s.u, TR, G(q + 4), G(q + 5), H, TR, false, B);
    STEP(o.linear(c.drh, H, s.tf1, nullptr, c.du, TR, H, TR, false, B));
    STEP(o.ln_bwd(c, s.t, c.du, P[q + 2], s.s1, c.dr, B, c.dt, G(q + 2), G(q + 3), TR, false, B));
    batch[nb++] = o.wgrad(c.dt, TR, s.lead, N_LEAD * D, G(q), G(q + 1), TR, N_LEAD * D, false, B);
    STEP(o.linear(c.dt, TR, s.tp, nullptr, c.g5, N_LEAD * D, TR, N_LEAD * D, false, B));
    STEP(flush());
    // blocks, last first; g: gradient of the block's output rows
    const u16* g = c.g5;
    for (int i = n.L - 1; i >= 0; --i) {
        const auto& k = s.blk[i];
        const bool fin = i + 1 == n.L;
        q = n.p_blk(i);
        batch[nb++] = o.wgrad(g, D, k.hid, F, G(q + 14), G(q + 15), D, F, !fin, LB);
        STEP(o.linear(g, D, k.t2, nullptr, c.gm, F, D, F, !fin, LB, BSRL_ACT_NONE, nullptr, 0, k.hid, F));
        batch[nb++] = o.wgrad(c.gm, F, k.h2, D, G(q + 12), G(q + 13), F, D, !fin, LB);
        STEP(o.linear(c.gm, F, k.t0, nullptr, c.dm, D, F, D, !fin, LB));
        STEP(o.ln_bwd(c, k.xm, c.dm, P[q + 10], k.s2, g, n.R, c.xm, G(q + 10), G(q + 11), D, !fin, LB));
        batch[nb++] = o.wgrad(c.xm, D, k.att, D, G(q + 8), G(q + 9), D, D, !fin, LB);
        STEP(o.linear(c.xm, D, k.to, nullptr, c.dm, D, D, D, !fin, LB));
        if (fin) {
            const AttnHeadsApart apart{s.apart, k.qkv, k.qkv + n.R * D, LB * (D / n.d.n_heads), n.R * (D / n.d.n_heads)};
            STEP(o.attn_bwd(k.q, D, k.qkv, k.qkv + D, 2 * D, s, c.dm, c.dq5, c.dqkv, c.dqkv + D, N_LEAD, either ? &apart : nullptr));
            batch[nb++] = o.wgrad(c.dqkv, 2 * D, k.h, D, G(q + 4), G(q + 5), 2 * D, D, true, 0);
            batch[nb++] = o.wgrad(c.dq5, D, k.h, D, G(q + 2), G(q + 3), D, D, false, LB);
            STEP(o.linear(c.dqkv, 2 * D, k.tqkv, nullptr, c.dm, D, 2 * D, D, true, 0));
            STEP(o.linear(c.dq5, D, k.tq, nullptr, c.dm, D, D, D, false, LB, BSRL_ACT_NONE, c.dm, D));
            STEP(flush());
            // the residual reaches the lead rows only; the critic's branch of the same stream joins behind it
            STEP(o.ln_bwd(c, k.x, c.dm, P[q], k.s1, c.xm, LB, c.dqkv, G(q), G(q + 1), D, true, 0));
            const int qc = n.p_critic();
            STEP(o.ln_bwd(c, last.x, c.gx, P[qc], s.sc, c.dqkv, n.R, c.g, G(qc), G(qc + 1), D, true, 0));
        } else {
            const AttnHeadsApart apart{s.apart, k.qkv + n.R * D, k.qkv + 2 * n.R * D, n.R * (D / n.d.n_heads), n.R * (D / n.d.n_heads)};
            STEP(o.attn_bwd(k.qkv, 3 * D, k.qkv + D, k.qkv + 2 * D, 3 * D, s, c.dm, c.dqkv, c.dqkv + D, c.dqkv + 2 * D, 0, either ? &apart : nullptr));
            batch[nb++] = o.wgrad(c.dqkv, 3 * D, k.h, D, G(q + 2), G(q + 3), 3 * D, D, true, 0);
            STEP(o.linear(c.dqkv, 3 * D, k.tqkv, nullptr, c.dm, D, 3 * D, D, true, 0));
            STEP(flush());
            STEP(o.ln_bwd(c, k.x, c.dm, P[q], k.s1, c.xm, n.R, c.g, G(q), G(q + 1), D, true, 0));
        }
        g = c.g;
    }
    // encoders: saber and leg tokens are two rows of an env's five
    o.copy(c.es, D, g, D, 2, N_LEAD * D, 2 * B, D);
    o.copy(c.el, D, g + 3 * D, D, 2, N_LEAD * D, 2 * B, D);
    const u16* dys[4] = {c.es, g + 2 * D, c.el, g + LB * D};
    for (int e = 0; e < 4; ++e) {
        const auto& k = s.enc[e];
        const int64_t rows = B * ENC_ROWS[e], ld = e == 1 ? N_LEAD * D : D;
        const int32_t* ex = e == 3 ? s.noff + B : nullptr;
        q = 4 * e;
        batch[nb++] = {dys[e], ld, k.hid, D, G(q + 2), G(q + 3), rows, ex, 0, D, D, D, D};
        LinArgs a{dys[e], ld, k.t2, nullptr, nullptr, 0, c.eh[e], D, nullptr, 0, 0, rows, (int)D, (int)D, 0, 0, 0, k.hid, D};
        a.extra = ex;
        STEP(bsrl_linear_run(a, BSRL_ACT_NONE, n.d.dtype, n.d.dtype, st, "bsrl_note_train"));
        batch[nb++] = {c.eh[e], D, k.in, PITCH, G(q), G(q + 1), rows, ex, 0, D, PITCH, D, n.enc_in(e)};
    }
    return flush();
}
#undef STEP

}  // namespace

extern "C" int64_t bsrl_note_train_layout(const bsrl_note_desc* d, int64_t* offsets, int64_t n_params) {
    if (!desc_ok(d) || !offsets) return 0;
    const Net n(*d, 1);
    return n_params == n.n_params() ? n.layout(offsets) : 0;
}

extern "C" int64_t bsrl_note_train_size(const bsrl_note_desc* d, int64_t B, int scratch) {
    if (!desc_ok(d) || B < 1 || B * (N_LEAD + N_NOTES) > 0x7fffffffLL) return 0;
    const Net n(*d, B);
    return (int64_t)(scratch ? Scratch(n, nullptr).bytes : n.saved(nullptr).bytes);
}

extern "C" int bsrl_note_train_forward(const bsrl_note_desc* d, const float* const* params, const void* obs, int64_t obs_ld, int obs_dtype,
                                       const int32_t* saber_idx, const int32_t* body_idx, float* vlogits, int64_t B, void* saved,
                                       int64_t saved_bytes, bsrl_stream stream) {
    if (!desc_ok(d)) return BSRL_UNSUPPORTED;
    if (!params || !obs || !saber_idx || !body_idx || !vlogits || B < 1) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_forward: bad argument");
    const int64_t need = bsrl_note_train_size(d, B, 0);
    if (!need || !saved || saved_bytes < need || !bsrl_aligned(saved, 256)) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_forward: workspace too small or unaligned");
    const Net n(*d, B);
    const Saved s = n.saved(static_cast<char*>(saved));
    hipStream_t st = static_cast<hipStream_t>(stream);
    int rc = front(n, s, params, obs, obs_ld, obs_dtype, saber_idx, body_idx, true, st);
    if (rc == BSRL_OK) rc = blocks(n, s, params, st);
    if (rc == BSRL_OK) rc = readout(n, s, params, vlogits, st);
    if (rc == BSRL_OK) BSRL_CHECK_LAUNCH("bsrl_note_train_forward");
    return rc;
}

bool note_train_saves(const bsrl_note_desc& d, int64_t B) {
    return desc_ok(&d) && bsrl_blocks_pair_saves(B, (int)d.d, d.n_heads, d.ffn, N_LEAD + N_NOTES, bsrl_cus());
}

extern "C" int bsrl_note_train_saves(const bsrl_note_desc* d, int64_t B) { return d && B >= 1 && note_train_saves(*d, B); }

BlocksSave note_train_blocks(const bsrl_note_desc& d, int64_t B, void* saved) {
    const Net n(d, B);
    const Saved s = n.saved(static_cast<char*>(saved));
    BlocksSave b = {s.noff, s.lead, (uint32_t)n.R, {}};
    for (int i = 0; i < n.L; ++i) {
        const auto& k = s.blk[i];
        b.blk[i] = {k.x, k.h, k.qkv, k.q, k.att, k.xm, k.h2, k.hid, k.s1.mean, k.s1.rstd, k.s2.mean, k.s2.rstd};
    }
    return b;
}

extern "C" int bsrl_note_train_begin(const bsrl_note_desc* d, const float* const* params, const void* obs, int64_t obs_ld, int obs_dtype,
                                     const int32_t* saber_idx, const int32_t* body_idx, int64_t B, void* saved, int64_t saved_bytes, bsrl_stream stream) {
    if (!d || !note_train_saves(*d, B)) return BSRL_UNSUPPORTED;
    if (!params || !obs || !saber_idx || !body_idx) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_begin: bad argument");
    if (!saved || saved_bytes < bsrl_note_train_size(d, B, 0) || !bsrl_aligned(saved, 256)) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_begin: workspace too small or unaligned");
    const Net n(*d, B);
    const int rc = front(n, n.saved(static_cast<char*>(saved)), params, obs, obs_ld, obs_dtype, saber_idx, body_idx, false, static_cast<hipStream_t>(stream));
    if (rc == BSRL_OK) BSRL_CHECK_LAUNCH("bsrl_note_train_begin");
    return rc;
}

extern "C" int bsrl_note_train_end(const bsrl_note_desc* d, const float* const* params, float* vlogits, int64_t B, void* saved, int64_t saved_bytes,
                                   bsrl_stream stream) {
    if (!d || !note_train_saves(*d, B)) return BSRL_UNSUPPORTED;
    if (!params || !vlogits) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_end: bad argument");
    if (!saved || saved_bytes < bsrl_note_train_size(d, B, 0) || !bsrl_aligned(saved, 256)) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_end: workspace too small or unaligned");
    const Net n(*d, B);
    const int rc = readout(n, n.saved(static_cast<char*>(saved)), params, vlogits, static_cast<hipStream_t>(stream));
    if (rc == BSRL_OK) BSRL_CHECK_LAUNCH("bsrl_note_train_end");
    return rc;
}

extern "C" int bsrl_note_train_backward(const bsrl_note_desc* d, const float* const* params, const float* dlogits, const float* dvlogits, float* grads,
                                        int64_t B, void* saved, int64_t saved_bytes, void* scratch, int64_t scratch_bytes, bsrl_stream stream) {
    if (!desc_ok(d)) return BSRL_UNSUPPORTED;
    if (!params || !dlogits || !dvlogits || !grads || B < 1) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_backward: bad argument");
    if (!saved || saved_bytes < bsrl_note_train_size(d, B, 0) || !bsrl_aligned(saved, 256) || !scratch || scratch_bytes < bsrl_note_train_size(d, B, 1) ||
        !bsrl_aligned(scratch, 256) || bsrl_note_train_size(d, B, 0) == 0) BSRL_FAIL(BSRL_EINVAL, "bsrl_note_train_backward: workspace too small or unaligned");
    const Net n(*d, B);
    int64_t off[16 + 16 * BSRL_MAX_LAYERS + 10 + 2 * N_HEADS_ACT + 16];
    n.layout(off);
    const Saved s = n.saved(static_cast<char*>(saved));
    const Scratch c(n, static_cast<char*>(scratch));
    const int rc = backward(n, s, c, params, dlogits, dvlogits, grads, off, static_cast<hipStream_t>(stream));
    if (rc == BSRL_OK) BSRL_CHECK_LAUNCH("bsrl_note_train_backward");
    return rc;
}

// (its name in ABI 22, when it took the one layout of q, k, v and bsrl_note_train_backward the other)
extern "C" int bsrl_note_train_stack_backward(const bsrl_note_desc* d, const float* const* params, const float* dlogits, const float* dvlogits, float* grads,
                                              int64_t B, void* saved, int64_t saved_bytes, void* scratch, int64_t scratch_bytes, bsrl_stream stream) {
    return bsrl_note_train_backward(d, params, dlogits, dvlogits, grads, B, saved, saved_bytes, scratch, scratch_bytes, stream);
}
