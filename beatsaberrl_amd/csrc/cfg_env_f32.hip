// The benchmark-config forward in fp32 (d = 128, 4 heads, F = 512, T <= 16), final block pruned to token 0, in ONE launch: one or
// two envs per workgroup of eight waves, their rows in LDS from the tokenizer to the logits.
//
// One kernel per op was a train of 20 dependent launches of 4 - 13 us whose Linears kept the matrix pipe a third busy: 113 us at 256
// envs, two blocks.  An env's 16 token rows are one MFMA tile, so here wave w owns feature tile w (and w + 8, ...) of every projection:
// its weight fragments are read by no other wave and go from L2 straight into registers, a group of eight in use and two in flight (64
// KB each per CU).  An output tile of v_mfma_f32_16x16x4 (lane: four features of one row) is the operand fragment of the next product
// as it stands, so the stream, LayerNorm's output, q | k, attention's output and the hidden cross LDS without a change of layout; V is
// computed with the operands' roles swapped, which lays it out over keys.  The weights come as an image of fragments: read in
// nn.Linear's layout a fragment is 16 rows of 64 bytes, and the same kernel took 58 us for 42.
// Behind the final block's keys and values only token 0 counts: matrix-vector products on the VALU, sixteenfold less work than
// tiles with one live row, bound by the weight stream.
// Bound: 900 MFMAs per SIMD and env at 32 cycles (12 us at two blocks), the weights (1.6 MB per workgroup out of L2, which a
// second env shares) and seven barriers per block.  Two blocks, launches -> this: 1 env 91 -> 37 us, 256 envs 113 -> 42, 512 143 -> 69.
// Arithmetic: products and sums in fp32, LayerNorm in two passes, expf / erff / exact division, as the launches that it replaces;
// distance to the model in 64 bits 3.3e-7 (they: 4.2e-7).
#include "block_stage.h"
#include "cfg_env_f32.h"

namespace {

constexpr int D = 128, NT = 8, KC = 8, H = 4, F = 512, NTHR = 512, NG = 12;      // NG: groups of KC fragments per block and wave
constexpr int ENV = 2 * NT * 64 + 4 * NT * 64, ROWS = 3 * D + F;                  // an env's fragments (float4), its single rows (floats)
constexpr int LN1G = 0, LN1B = D, BQKV = 2 * D, BO = 5 * D, LN2G = 6 * D, LN2B = 7 * D, B1 = 8 * D, B2 = 8 * D + F, LV = 9 * D + F;
constexpr size_t lds_bytes(int r, int layers) { return (size_t)r * (ENV * 16 + ROWS * 4) + (size_t)layers * LV * 4; }

__device__ __forceinline__ f32x4 mma4(const f32x4& a, const f32x4& b, f32x4 c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
}
__device__ __forceinline__ float sum_rows(float v) { float u = v; rows_reduce2(v, u, OpAdd()); return v; }

// The weight image, in fragments of 64 lanes x 4 floats: fragment (tile t, chunk c) of a matrix holds W[16 t + lane % 16][16 c + 4 (lane
// / 16) + 0..3], zero past its rows and columns.  prop | obj | per block q | k | v, output projection, W1, W2 | heads, tile by tile.
constexpr int BLK_FRAGS = (3 * NT + NT + F / 16) * KC + NT * (F / 16);
struct Image {
    int obj, blk, heads, head_tiles, prop_chunks, obj_chunks, total;
    __host__ __device__ Image(int prop_dim, int obj_dim, int layers, int n_out) {
        prop_chunks = (prop_dim + 15) / 16; obj_chunks = (obj_dim + 15) / 16; head_tiles = (n_out + 15) / 16;
        obj = NT * prop_chunks; blk = obj + NT * obj_chunks; heads = blk + layers * BLK_FRAGS; total = heads + head_tiles * KC;
    }
};
// one wave per fragment
__global__ __launch_bounds__(256) void cfg_env_f32_pack_kernel(bsrl_cfg_rows_weights w, f32x4* img, int prop_dim, int obj_dim, int layers, int n_out) {
    const Image im(prop_dim, obj_dim, layers, n_out);
    const int f = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (f >= im.total) return;
    const void* src; int r, chunks = KC, K = D, rows = 1 << 30;      // r: the fragment inside its matrix
    if (f < im.obj) { src = w.prop_w; r = f; chunks = im.prop_chunks; K = prop_dim; }
    else if (f < im.blk) { src = w.obj_w; r = f - im.obj; chunks = im.obj_chunks; K = obj_dim; }
    else if (f >= im.heads) { src = w.heads_w; r = f - im.heads; rows = n_out; }
    else {
        const auto& k = w.blk[(f - im.blk) / BLK_FRAGS];
        r = (f - im.blk) % BLK_FRAGS;
        if (r < 3 * NT * KC) src = k.qkv_w;
        else if (r < 4 * NT * KC) { src = k.out_w; r -= 3 * NT * KC; }
        else if (r < 8 * NT * KC) { src = k.w0; r -= 4 * NT * KC; }
        else { src = k.w2; r -= 8 * NT * KC; chunks = F / 16; K = F; }
    }
    const int row = 16 * (r / chunks) + (lane & 15), k0 = 16 * (r % chunks) + 4 * (lane >> 4);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (row < rows) {
        const float* p = static_cast<const float*>(src) + (int64_t)row * K + k0;
#pragma unroll
        for (int j = 0; j < 4; ++j) if (k0 + j < K) v[j] = p[j];
    }
    img[(int64_t)f * 64 + lane] = v;
}

// R: envs per workgroup
template <int ACT, int R>
__global__ __launch_bounds__(NTHR, 2) void cfg_env_f32_kernel(CfgEnvF32Args a) {
    extern __shared__ __attribute__((aligned(16))) f32x4 lds[];
    f32x4* const xs = lds;                           // residual stream [env][feature tile][lane]
    f32x4* const hs = xs + R * NT * 64;              // LayerNorm output
    f32x4* const un = hs + R * NT * 64;              // per env q | k | v | attention's output, then the hidden
    constexpr int UN = 4 * NT * 64;
    float* const rows = reinterpret_cast<float*>(un + R * UN);        // token 0 of the final block, per env: q | attention | x | hidden
    float* const vecs = rows + R * ROWS;             // every block's vectors
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int L = a.n_layers, ngrp = (a.B + R - 1) / R;
    const Image im(a.prop_dim, a.obj_dim, L, a.n_out);
    const float scale = 0.17677669529663688110f;     // 1 / sqrt(32)

    // the vectors, 64 floats of one of them per wave and load, four loads in flight
    for (int s0 = w; s0 < L * (LV / 64); s0 += 32) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            int s = s0 + 8 * u;
            s = s < L * (LV / 64) ? s : 0;
            const int l = s / (LV / 64), r = (s - l * (LV / 64)) * 64;
            const auto& k = a.w.blk[l];
            const float* p = r < LN1B ? k.ln_attn_w + r : r < BQKV ? k.ln_attn_b + (r - LN1B) : r < BO ? k.qkv_b + (r - BQKV) : r < LN2G ? k.out_b + (r - BO) :
                             r < LN2B ? k.ln_ffn_w + (r - LN2G) : r < B1 ? k.ln_ffn_b + (r - LN2B) : r < B2 ? k.b0 + (r - B1) : k.b2 + (r - B2);
            v[u] = p[tid & 63];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) if (s0 + 8 * u < L * (LV / 64)) vecs[(s0 + 8 * u) * 64 + (tid & 63)] = v[u];
    }
    for (int grp = blockIdx.x; grp < ngrp; grp += gridDim.x) {
        int lane = tid & 63;
        asm("" : "+v"(lane));                        // a value of this iteration: a hundred addresses are not kept over all of them
        const int r16 = lane & 15, g = lane >> 4;
        // KC fragments of the image from fragment `at` on
        auto load_at = [&](f32x4 (&f)[KC], int at) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            const f32x4* p = static_cast<const f32x4*>(a.w.lead_img) + (int64_t)at * 64;
#pragma unroll
            for (int c = 0; c < KC; ++c) f[c] = p[c * 64 + lane];
            __builtin_amdgcn_sched_barrier(0);
        };
        // group gi of block l: q, k, v; output projection; W1's tiles w + 8 i; W2 in k quarters
        auto load = [&](f32x4 (&f)[KC], int l, auto gi_) __attribute__((always_inline)) {
            constexpr int gi = decltype(gi_)::value;
            load_at(f, im.blk + l * BLK_FRAGS + (gi < 8 ? (gi * NT + w) * KC : 8 * NT * KC + (w * 4 + gi - 8) * KC));
        };
        auto load_heads = [&](f32x4 (&f)[KC], int tile) __attribute__((always_inline)) { load_at(f, im.heads + (tile < im.head_tiles ? tile : 0) * KC); };
        auto at4 = [&](const float* p) __attribute__((always_inline)) { return *reinterpret_cast<const f32x4*>(p + 4 * g); };
        const int env0 = grp * R;
        auto env_of = [&](int e) __attribute__((always_inline)) { return env0 + e < a.B ? env0 + e : a.B - 1; };      // past the end: not stored
        f32x4 buf[3][KC];
        auto first = [&] __attribute__((always_inline)) {
            static_for<0, 3>([&](auto i) __attribute__((always_inline)) { load(buf[decltype(i)::value], 0, i); });
        };
        if constexpr (R == 1) first();               // (two envs' observations leave no room for them in registers)
        int lim[R];                                  // the last key that is looked at, whatever those past it hold
#pragma unroll
        for (int e = 0; e < R; ++e) {
            const int nv = a.n_valid ? a.n_valid[env_of(e)] : a.T - 1;
            lim[e] = nv < 0 ? 0 : nv < a.T ? nv : a.T - 1;
        }
        // ---- tokenizer: row 0 from the proprio block, the others from their object, one accumulator ----
        f32x4 x[R];                                  // this wave's feature tile
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float b = (r16 == 0 ? a.w.prop_b : a.w.obj_b)[16 * w + 4 * g + i];
#pragma unroll
            for (int e = 0; e < R; ++e) x[e][i] = b;
        }
        auto embed = [&](int frag, int chunks, int K, bool on, int64_t at) __attribute__((always_inline)) {
            constexpr int EC = 4;                    // chunks of 16 k at a time
            for (int c0 = 0; c0 < chunks; c0 += EC) {
                f32x4 wf[EC], of[R][EC];
#pragma unroll
                for (int c = 0; c < EC; ++c) {
                    const int cc = c0 + c < chunks ? c0 + c : 0;
                    wf[c] = static_cast<const f32x4*>(a.w.lead_img)[(int64_t)(frag + w * chunks + cc) * 64 + lane];
#pragma unroll
                    for (int e = 0; e < R; ++e)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int k = 16 * (c0 + c) + 4 * g + j;
                            const bool in = on && k < K;
                            const float o = a.obs[env_of(e) * a.obs_ld + (in ? at + k : 0)];
                            of[e][c][j] = in ? o : 0.f;
                        }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < EC; ++c)
                    if (c0 + c < chunks)
#pragma unroll
                        for (int e = 0; e < R; ++e) x[e] = mma4(wf[c], of[e][c], x[e]);
            }
        };
        embed(0, im.prop_chunks, a.prop_dim, r16 == 0, 0);
        embed(im.obj, im.obj_chunks, a.obj_dim, r16 >= 1 && r16 < a.T, a.prop_dim + (int64_t)(r16 - 1) * a.obj_dim);
        if constexpr (R > 1) first();
        auto keep_x = [&] __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < R; ++e) xs[(e * NT + w) * 64 + lane] = x[e];
        };
        keep_x();
        blk_barrier();

        // (v - mean) * rstd * gamma + beta of a row whose features 16 c + 4 g + i this lane holds
        auto stats = [&](const f32x4 (&v)[NT], float& mean, float& rstd) __attribute__((always_inline)) {
            float s = 0.f, q = 0.f;
#pragma unroll
            for (int c = 0; c < NT; ++c) s += (v[c][0] + v[c][1]) + (v[c][2] + v[c][3]);
            mean = sum_rows(s) * (1.0f / D);
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) { const float t = v[c][i] - mean; q = fmaf(t, t, q); }
            rstd = 1.0f / sqrtf(sum_rows(q) * (1.0f / D) + 1e-5f);
        };
        auto norm = [&](const float* gamma, const float* beta) __attribute__((always_inline)) {
            const int e = R == 1 ? 0 : w >> 2;                   // each wave forms its env's statistics and writes R of the eight tiles
            f32x4 v[NT];
#pragma unroll
            for (int c = 0; c < NT; ++c) v[c] = xs[(e * NT + c) * 64 + lane];
            float mean, rstd;
            stats(v, mean, rstd);
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int t = R == 1 ? w : 2 * (w & 3) + k;
                const f32x4 u = xs[(e * NT + t) * 64 + lane], gm = at4(gamma + 16 * t), bt = at4(beta + 16 * t);
                f32x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = (u[i] - mean) * rstd * gm[i] + bt[i];
                hs[(e * NT + t) * 64 + lane] = o;
            }
            blk_barrier();
        };
        f32x4 act[R][KC];                            // the other operand of a group, read from LDS in one burst
        auto get = [&](const f32x4* p, int pitch) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 0; e < R; ++e)
#pragma unroll
                for (int c = 0; c < KC; ++c) act[e][c] = p[e * pitch + c * 64 + lane];
            __builtin_amdgcn_sched_barrier(0);
        };
        auto mma = [&](const f32x4 (&f)[KC], f32x4 (&acc)[R]) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < KC; ++c)
#pragma unroll
                for (int e = 0; e < R; ++e) acc[e] = mma4(f[c], act[e][c], acc[e]);
        };

        // group gi of block l has had its last use: the group three behind it takes its place (behind the final block: the readout's tiles w, w + 8)
        auto next = [&](auto gi_, int l, auto fin) __attribute__((always_inline)) {
            constexpr int gi = decltype(gi_)::value + 3;
            if constexpr (gi < NG) load(buf[gi % 3], l, std::integral_constant<int, gi>{});
            else if constexpr (!decltype(fin)::value) load(buf[gi % 3], l + 1, std::integral_constant<int, gi % NG>{});
            else if constexpr (gi % NG < 2) load_heads(buf[gi % 3], w + NT * (gi % NG));
        };
        typedef std::false_type Full;
        typedef std::true_type Final;
        auto project = [&](auto t_, int l, auto fin) __attribute__((always_inline)) {       // part t of q | k | v, this wave's tile
            const float* lv = vecs + l * LV;
            constexpr int t = decltype(t_)::value;
            f32x4 acc[R];
            if constexpr (t < 2) {
                const f32x4 b = at4(lv + BQKV + D * t + 16 * w);
#pragma unroll
                for (int e = 0; e < R; ++e) acc[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
                mma(buf[t], acc);
#pragma unroll
                for (int e = 0; e < R; ++e) acc[e] += b;
            } else {                             // V over keys: operand roles swapped
                const float b = lv[BQKV + 2 * D + 16 * w + r16];
#pragma unroll
                for (int e = 0; e < R; ++e) {
                    acc[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int c = 0; c < KC; ++c) acc[e] = mma4(act[e][c], buf[2][c], acc[e]);
                    acc[e] += b;
                }
            }
            next(t_, l, fin);
#pragma unroll
            for (int e = 0; e < R; ++e) un[e * UN + (t * NT + w) * 64 + lane] = acc[e];
        };
        // attention of one head: keys 4 g + i of query r16 in a lane
        auto attend = [&](int e, int hd, const f32x4 (&qf)[2], int last, f32x4 (&o)[2]) __attribute__((always_inline)) {
            const f32x4* kp = un + e * UN + (NT + 2 * hd) * 64 + lane;
            f32x4 s = {0.f, 0.f, 0.f, 0.f}, v[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) { s = mma4(kp[c * 64], qf[c], s); v[c] = kp[(NT + c) * 64]; }
            float m = -INFINITY, sum = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool in = 4 * g + i <= last;
                s[i] = in ? s[i] * scale : -INFINITY;
                v[0][i] = in ? v[0][i] : 0.f; v[1][i] = in ? v[1][i] : 0.f;
                m = fmaxf(m, s[i]);
            }
            float m1 = m;
            rows_reduce2(m, m1, OpMax());
#pragma unroll
            for (int i = 0; i < 4; ++i) { s[i] = expf(s[i] - m); sum += s[i]; }
            const float inv = 1.0f / sum_rows(sum);
#pragma unroll
            for (int c = 0; c < 2; ++c) o[c] = mma4(v[c], s, (f32x4){0.f, 0.f, 0.f, 0.f}) * inv;
        };
        const int ae = R == 1 ? 0 : w >> 2, ah = w & 3;      // the env and head whose attention this wave does
        const bool attends = R > 1 || w < 4;
        int alim = lim[0];
        if (R > 1 && ae == 1) alim = lim[R - 1];
        for (int l = 0; l + 1 < L; ++l) {
            const float* lv = vecs + l * LV;
            norm(lv + LN1G, lv + LN1B);
            get(hs, NT * 64);
            static_for<0, 3>([&](auto t_) __attribute__((always_inline)) { project(t_, l, Full()); });
            blk_barrier();
            if (attends) {
                f32x4 qf[2], o[2];
#pragma unroll
                for (int c = 0; c < 2; ++c) qf[c] = un[ae * UN + (2 * ah + c) * 64 + lane];
                attend(ae, ah, qf, alim, o);
#pragma unroll
                for (int c = 0; c < 2; ++c) un[ae * UN + (3 * NT + 2 * ah + c) * 64 + lane] = o[c];
            }
            blk_barrier();
            // ---- output projection onto the residual ----
            f32x4 acc[R];
            auto onto_x = [&](const float* bias) __attribute__((always_inline)) {
                const f32x4 b = at4(bias + 16 * w);
#pragma unroll
                for (int e = 0; e < R; ++e) x[e] += acc[e] + b;
                keep_x();
                blk_barrier();
            };
            get(un + 3 * NT * 64, UN);
#pragma unroll
            for (int e = 0; e < R; ++e) acc[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
            mma(buf[0], acc);
            next(std::integral_constant<int, 3>{}, l, Full());
            onto_x(lv + BO);
            // ---- LayerNorm + FFN ----
            norm(lv + LN2G, lv + LN2B);
            get(hs, NT * 64);
            static_for<0, 4>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                const int t = w + NT * i;
                const f32x4 b = at4(lv + B1 + 16 * t);
#pragma unroll
                for (int e = 0; e < R; ++e) acc[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
                mma(buf[(4 + i) % 3], acc);
                next(std::integral_constant<int, 4 + i>{}, l, Full());
#pragma unroll
                for (int e = 0; e < R; ++e) {
                    f32x4 h;
#pragma unroll
                    for (int j = 0; j < 4; ++j) h[j] = apply_act<ACT>(acc[e][j] + b[j]);
                    un[e * UN + t * 64 + lane] = h;
                }
            });
            blk_barrier();
#pragma unroll
            for (int e = 0; e < R; ++e) acc[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
            static_for<0, 4>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value;
                get(un + KC * i * 64, UN);
                mma(buf[(8 + i) % 3], acc);
                next(std::integral_constant<int, 8 + i>{}, l, Full());
            });
            onto_x(lv + B2);
        }
        const float* lv = vecs + (L - 1) * LV;
        norm(lv + LN1G, lv + LN1B);
        get(hs, NT * 64);
        // ---- the final block: keys and values of every row, then token 0 alone, a column per lane (its k over the four g) ----
        auto row_of = [&](int e, int at) __attribute__((always_inline)) { return rows + e * ROWS + at; };
        constexpr int RQ = 0, RA = D, RX = 2 * D, RH = 3 * D;
        auto dot = [&](const f32x4 (&f)[KC], const f32x4 (&v)[KC]) __attribute__((always_inline)) {
            f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < KC; ++c)
#pragma unroll
                for (int j = 0; j < 4; ++j) s[j] = fmaf(f[c][j], v[c][j], s[j]);
            return sum_rows((s[0] + s[1]) + (s[2] + s[3]));
        };
        auto read = [&](f32x4 (&v)[KC], const float* p) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < KC; ++c) v[c] = at4(p + 16 * c);
        };
        f32x4 v[KC];
#pragma unroll
        for (int e = 0; e < R; ++e) {
#pragma unroll
            for (int c = 0; c < KC; ++c) v[c] = hs[(e * NT + c) * 64 + 16 * g];
            const float q = dot(buf[0], v) + lv[BQKV + 16 * w + r16];
            if (g == 0) row_of(e, RQ)[16 * w + r16] = q;
        }
        next(std::integral_constant<int, 0>{}, L - 1, Final());
        static_for<1, 3>([&](auto t_) __attribute__((always_inline)) { project(t_, L - 1, Final()); });
        blk_barrier();
        if (attends) {
            f32x4 qf[2], o[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) qf[c] = at4(row_of(ae, RQ) + 32 * ah + 16 * c);
            attend(ae, ah, qf, alim, o);
            if (r16 == 0) {
#pragma unroll
                for (int c = 0; c < 2; ++c) *reinterpret_cast<f32x4*>(row_of(ae, RA) + 32 * ah + 16 * c + 4 * g) = o[c];
            }
        }
        blk_barrier();
        float x0[R];                             // feature 16 w + r16 of token 0
#pragma unroll
        for (int e = 0; e < R; ++e) {
            read(v, row_of(e, RA));
            x0[e] = reinterpret_cast<const float*>(xs + (e * NT + w) * 64 + 16 * (r16 >> 2))[r16 & 3];
            x0[e] += dot(buf[0], v) + lv[BO + 16 * w + r16];
            if (g == 0) row_of(e, RX)[16 * w + r16] = x0[e];
        }
        next(std::integral_constant<int, 3>{}, L - 1, Final());
        blk_barrier();
        auto norm_row = [&](const float* p, const float* gamma, const float* beta) __attribute__((always_inline)) {      // every wave its own copy
            read(v, p);
            float mean, rstd;
            stats(v, mean, rstd);
#pragma unroll
            for (int c = 0; c < KC; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) v[c][i] = (v[c][i] - mean) * rstd * gamma[16 * c + 4 * g + i] + beta[16 * c + 4 * g + i];
        };
#pragma unroll
        for (int e = 0; e < R; ++e) {
            norm_row(row_of(e, RX), lv + LN2G, lv + LN2B);
#pragma unroll
            for (int c = 0; c < KC; ++c) act[e][c] = v[c];
        }
        static_for<0, 4>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            const int col = 16 * (w + NT * i) + r16;
#pragma unroll
            for (int e = 0; e < R; ++e) {
                const float h = apply_act<ACT>(dot(buf[(4 + i) % 3], act[e]) + lv[B1 + col]);
                if (g == 0) row_of(e, RH)[col] = h;
            }
            next(std::integral_constant<int, 4 + i>{}, L - 1, Final());
        });
        blk_barrier();
        float y[R] = {};
        static_for<0, 4>([&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
#pragma unroll
            for (int e = 0; e < R; ++e) { read(v, row_of(e, RH) + D * i); y[e] += dot(buf[(8 + i) % 3], v); }
            next(std::integral_constant<int, 8 + i>{}, L - 1, Final());
        });
#pragma unroll
        for (int e = 0; e < R; ++e) if (g == 0) row_of(e, RX)[16 * w + r16] = x0[e] + (y[e] + lv[B2 + 16 * w + r16]);
        blk_barrier();
        // ---- readout: 29 K logits + value, output tiles w, w + 8, ... ----
#pragma unroll
        for (int e = 0; e < R; ++e) {
            if (a.final_ln) norm_row(row_of(e, RX), a.w.final_ln_w, a.w.final_ln_b);
            else read(v, row_of(e, RX));
#pragma unroll
            for (int c = 0; c < KC; ++c) act[e][c] = v[c];
        }
        auto head = [&](const f32x4 (&f)[KC], int tile) __attribute__((always_inline)) {
            const int col = 16 * tile + r16;
#pragma unroll
            for (int e = 0; e < R; ++e) {
                const float o = dot(f, act[e]);
                if (g == 0 && col < a.n_out && env0 + e < a.B) {
                    const float b = o + a.w.heads_b[col];
                    if (col + 1 < a.n_out) a.logits[(int64_t)(env0 + e) * (a.n_out - 1) + col] = b;
                    else a.value[env0 + e] = b;
                }
            }
        };
        head(buf[0], w);
        head(buf[1], w + NT);
        for (int tile = w + 2 * NT; 16 * tile < a.n_out; tile += NT) { load_heads(buf[2], tile); head(buf[2], tile); }
    }
}

template <int ACT, int R>
bool launch(const CfgEnvF32Args& a, int cus, hipStream_t st) {
    auto kern = cfg_env_f32_kernel<ACT, R>;
    const size_t dyn = lds_bytes(R, a.n_layers);
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    const int n = (a.B + R - 1) / R;
    hipLaunchKernelGGL(kern, dim3((unsigned)(n < cus ? n : cus)), dim3(NTHR), dyn, st, a);
    return true;
}
template <int ACT>
bool by_batch(const CfgEnvF32Args& a, hipStream_t st) {
    const int cus = bsrl_cus();
    return a.B <= cus ? launch<ACT, 1>(a, cus, st) : launch<ACT, 2>(a, cus, st);
}

}  // namespace

int64_t bsrl_cfg_env_f32_pack_size(const bsrl_cfg_desc* d) {
    static_assert(lds_bytes(2, BSRL_MAX_LAYERS) <= (size_t)LDS_BUDGET, "two envs and every block's vectors fit a workgroup's LDS");
    if (d->dtype != BSRL_F32 || d->d != D || d->n_heads != H || d->ffn != F || d->T > 16 || d->prop_dim > 4096 || d->obj_dim > 64 || d->n_gears > 64) return 0;
    return (int64_t)Image(d->prop_dim, d->obj_dim, d->n_layers, 29 * d->n_gears + 1).total * 1024;
}
int bsrl_cfg_env_f32_pack(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w, void* img, hipStream_t st) {
    const int n_out = 29 * d->n_gears + 1, total = Image(d->prop_dim, d->obj_dim, d->n_layers, n_out).total;
    hipLaunchKernelGGL(cfg_env_f32_pack_kernel, dim3((unsigned)((total + 3) / 4)), dim3(256), 0, st, *w, static_cast<f32x4*>(img), d->prop_dim, d->obj_dim,
                       d->n_layers, n_out);
    BSRL_CHECK_LAUNCH("bsrl_cfg_rows_pack");
    return BSRL_OK;
}
bool bsrl_cfg_env_f32(const bsrl_cfg_desc* d, const CfgEnvF32Args& a, hipStream_t st) {
    return d->act == BSRL_ACT_GELU ? by_batch<BSRL_ACT_GELU>(a, st) : by_batch<BSRL_ACT_RELU>(a, st);
}
