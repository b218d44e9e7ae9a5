// Argument block shared by the linear kernels.
#pragma once
#include "bsrl_common.h"

struct LinArgs {
    const void* x; int64_t ldx;
    const void* w;
    const float* bias;
    const void* res; int64_t ldr;
    void* y; int64_t ldy;
    void* y2; int64_t ldy2; int64_t split;
    int64_t rows; int K; int M;
    int out_f32;
    // grouped output rows (0 = off): output row r lives at (r / y_group) * y_gstride + (r % y_group) * ldy,
    // i.e. y is a (rows / y_group, y_group, M) view of a larger tensor (a token slice of a (B, T, d) stream)
    int y_group; int64_t y_gstride;
    // ReLU gate (NULL = off): the result is kept where gate[row * ldgate + col] > 0 and zeroed elsewhere - the
    // backward of a ReLU whose forward output is `gate`, applied in the epilogue of the data-gradient GEMM
    const void* gate; int64_t ldgate;
    // rows counted on the device: base + *extra of them, `rows` their host-side bound (NULL: exactly `rows`)
    const int32_t* extra = nullptr; int64_t base = 0;
    bool vec_ok = false;               // linear_small.hip: filled in by its launch
    bool res_f32 = false;              // 16-bit operands with an fp32 residual, no activation (linear_small.hip alone)
};

__device__ __forceinline__ int64_t lin_rows(const LinArgs& a) { return a.extra ? a.base + (int64_t)*a.extra : a.rows; }

// element offset of output row `row` in y (rows < 2^31 is checked on the host)
__device__ __forceinline__ int64_t lin_yoff(const LinArgs& a, int64_t row) {
    if (a.y_group == 0) return row * a.ldy;
    const uint32_t r = (uint32_t)row, gq = r / (uint32_t)a.y_group;
    return (int64_t)gq * a.y_gstride + (int64_t)(r - gq * (uint32_t)a.y_group) * a.ldy;
}

// LDS-tiled 16-bit kernel for large row counts (linear_tiled.hip); returns false when the
// shape is outside what it covers (the caller then takes the direct-from-global kernel).
bool bsrl_linear_tiled(const LinArgs& a, int act, int dtype, hipStream_t st);

// Weight-resident streaming 16-bit kernel for many rows and K = 128 / 192 / 256 / 384 (linear_stream.hip);
// false when the shape is outside what it covers.
bool bsrl_linear_stream(const LinArgs& a, int act, int dtype, hipStream_t st);

// Two Linears with a ReLU between them in one launch (linear_stream.hip): x (rows, K1) -> relu(x W1^T + b1) -> l2 (its
// w, bias, y, grouping, rows; K = M = d), up to MLP2_MAX problems of one d at once; false when the shape is outside what it
// covers (K1 = 64, d = 128 / 192, 16-bit).
struct Mlp2Args {
    LinArgs l2;
    const void* x; int64_t ldx;           // (rows, K1) 16-bit
    const void* w1; const float* b1;      // (d, K1) 16-bit, (d) fp32
};
constexpr int MLP2_MAX = 4;
bool bsrl_mlp2_stream(const Mlp2Args* a, int n, int64_t K1, int dtype, hipStream_t st);

// Ring-buffered 16-bit kernel for large row counts and K a multiple of 32 (linear_ring.hip): operands go from
// global memory straight into an LDS ring; false when the shape is outside what it covers.
bool bsrl_linear_ring(const LinArgs& a, int act, int dtype, hipStream_t st);

// Latency kernel for small row counts, and the fp32 path (linear_small.hip); false when K or the operands' alignment are
// outside what it covers.
bool bsrl_linear_small(const LinArgs& a, int act, int dtype, hipStream_t st);

// The dispatch behind bsrl_linear / bsrl_linear_gated (linear.hip), for host code that composes forwards and backwards.
int bsrl_linear_run(const LinArgs& a, int act, int dtype, int out_dtype, hipStream_t st, const char* what);

// LayerNorm of rows + *extra rows (ln.hip; `bound`: their host-side bound) at row pitches ldx, ldy; mean, rstd optional;
// x_f32: x is fp32 whatever dtype is y's
int bsrl_ln_rows(const void* x, int64_t ldx, const float* w, const float* b, void* y, int64_t ldy, float* mean, float* rstd, int64_t rows, const int32_t* extra,
                 int64_t bound, int64_t d, float eps, int dtype, bsrl_stream stream, bool x_f32 = false);

// The backward side over device-counted rows, for host code that composes a backward (ln_bwd.hip, wgrad.hip, attn_bwd.hip)
int bsrl_ln_bwd_rows(const void* x, const void* dy, const float* weight, const float* mean, const float* rstd, const void* gx,
                     int64_t gx_rows, void* dx, float* dw, float* db, float* dbb, void* workspace, int64_t rows, const int32_t* extra,
                     int64_t bound, int64_t d, int dtype, bsrl_stream stream);
// dW (MO, KO) = the leading part of dy^T x, dy (rows, M), x (rows, K): columns past MO / KO are the operands' padding.  rows: with
// `extra` the host-side bound of base + *extra.  Up to 12 problems at once; the workspace's size depends on shapes and rows only
// (operands 16-byte aligned, pitches multiples of 8).
struct WgradProblem {
    const void* dy; int64_t lddy; const void* x; int64_t ldx; float *dw, *db;
    int64_t rows; const int32_t* extra; int64_t base, M, K, MO, KO;
};
int64_t bsrl_wgrad_batch_size(const WgradProblem* p, int n);
int bsrl_wgrad_batch(const WgradProblem* p, int n, void* workspace, int64_t bytes, int dtype, bsrl_stream stream);
// A batch for which two forms are enqueued, of which the device takes one (cfg_rows.hip): per env, where its optional tokens are at most
// `most` (below) or more (not below).  Rows and envs of the per-env form and of the other; where they are 0 its kernels return at once.
struct RowsPick { int32_t own_rows, own_envs, rows, envs; };
int bsrl_token_offsets_pick(const int32_t* n_valid, int64_t B, int64_t opt, int32_t* noff, int64_t most, bool below, RowsPick* pick, bsrl_stream stream);
// bsrl_cfg_tokens, bsrl_attn_ragged; go: 0 or B (NULL: B)
int bsrl_cfg_tokens_if(const int32_t* go, const void* obs, int64_t obs_ld, int obs_dtype, const void* wp, const float* bp, const void* wo,
                       const float* bo, const int32_t* noff, void* tokens, int64_t B, int64_t d, int64_t prop_dim, int64_t obj_dim, int dtype,
                       bsrl_stream stream);
// bsrl_attn_ragged with the keys in the slots of the full stream (attn.hip; slots (B, 32), T <= 32, 16-bit)
int bsrl_attn_ragged_slots(const void* q, int64_t q_ld, const void* k, int64_t k_ld, const void* v, int64_t v_ld, const int32_t* noff,
                           const uint8_t* slots, const void* opt_bias, void* out, int64_t out_ld, int64_t B, int64_t lead, int64_t opt,
                           int64_t n_queries, int64_t H, int64_t dh, int dtype, bsrl_stream stream, const int32_t* go = nullptr);
bool bsrl_attn_bwd_ragged_ok(int64_t T, int64_t H, int64_t dh, int dtype);
// apart: where *flag (device) is not zero, q, k, v lie head after head, a head's rows one after another and the next head's q_hs | kv_hs
// elements on, k and v at these addresses; where it is zero as the other arguments say
struct AttnHeadsApart { const float* flag; const void *k, *v; int64_t q_hs, kv_hs; };
int bsrl_attn_bwd_ragged(const void* q, int64_t q_ld, const void* k, int64_t k_ld, const void* v, int64_t v_ld, const int32_t* noff,
                         const void* opt_bias, const void* dout, int64_t do_ld, void* dq, int64_t dq_ld, void* dk, int64_t dk_ld,
                         void* dv, int64_t dv_ld, int64_t B, int64_t lead, int64_t opt, int64_t nq, int64_t H, int64_t dh, int dtype,
                         bsrl_stream stream, const AttnHeadsApart* apart = nullptr);
// NotePolicy front end into the compacted stream (frontend.hip): counts of the attendable notes, then the padded encoder inputs
// with the note rows and their key bias at noff[b], and the token in each key slot (slots (B, 32), 255 = dropped)
int bsrl_note_counts(const void* obs, int64_t obs_ld, int obs_dtype, int32_t* counts, int64_t B, int dtype, bsrl_stream stream);
int bsrl_note_frontend_rows(const void* obs, int64_t obs_ld, int obs_dtype, const int32_t* saber_idx, const int32_t* body_idx,
                            int note_geo, int flux, float z_asinh, const int32_t* noff, void* saber_in, void* torso_in, void* leg_in,
                            void* note_in, void* note_bias, uint8_t* slots, int64_t B, int dtype, bsrl_stream stream);
