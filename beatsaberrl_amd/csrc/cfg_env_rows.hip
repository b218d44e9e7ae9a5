// The benchmark-config forward of few envs at d = 384 (12 heads of 32, F = 1536, T <= 48, 16 bit; final block pruned to token 0) in
// TWO launches per block.
//
// One kernel per op was 47 dependent launches of 4 - 14 us, of which a launch, a memory round trip and a few hundred cycles of MFMAs
// are what each has to do: 350 us at 97 envs, six blocks.  Here
//   * env_block_kernel: an env per workgroup of twelve waves, a head per wave.  The block's input rows (the former block's FFN parts
//     summed, or the tokenizer), LayerNorm, the head's q | k | v, its attention - all in the wave's registers -, output projection and
//     residual.  No other wave reads a wave's weight fragments: they go from L2 straight into its registers, sixteen ahead;
//   * env_ffn_kernel: 32 rows of the batch and a QUARTER of the hidden per workgroup (the weights are what a workgroup of all of them
//     would wait for: 2.4 MB at 64 B/clk), LayerNorm in its prologue; the four parts of the down-projection meet in the next launch's
//     prologue, in fixed order.
// 97 envs, a quarter of them empty: 350 -> 219 us; 1 env 242 -> 206, 234 envs 481 -> 274 (no mask 866 -> 484).  Bound: env_block 18 us (its
// rows 5, LayerNorm 2.5, q | k | v 5 at the 64 B/clk into a CU, attention 2, barriers 2), env_ffn 8 us (weights 5 at that rate).  What
// made the difference there: loads in the order in which they are wanted, as they retire in order; the vectors through LDS; one body
// for one to three row tiles (three bodies of straight-line code: + 4 us of instruction misses); no register spilled (+ 3 us).
// Fetching the next launch's weights into the L2s by extra workgroups gave 4 % at 97 envs and cost 9 % at 1 and at 234: not kept.
// Rows lie env by env: row j of env b is b + noff[b] + j; behind the final block row b is env b's token 0.
// Rounding points are those of the launches: the stream, LayerNorm's output, q | k | v, the probabilities, attention's output and the
// hidden once each; sums in fp32.
#include "block_stage.h"
#include "cfg_env_rows.h"

namespace {

constexpr int D = 384, NT = 24, KC = 12, H = 12, F = 4 * D, MT = 48, SL = 4;      // SL: slices of the hidden
constexpr int XLD = D + 8;                           // row pitch of the residual rows in LDS
constexpr int BLK_FRAGS = (3 * NT + NT + F / 16) * KC + NT * (F / 32), OUT_AT = 3 * NT * KC, W0_AT = 4 * NT * KC, W2_AT = W0_AT + (F / 16) * KC;

// The weight image, in fragments of 64 lanes x 16 bytes: fragment (tile t, chunk c) of a matrix holds W[16 t + lane % 16][32 c + k(lane
// / 16, 0..7)], zero past its rows and columns; k in order, or (output projection, W2: their operands are accumulator tiles in pairs)
// 4 g + 0..3 and 16 + 4 g + 0..3.  prop | obj | per block q | k | v, output projection, W1, W2 | heads, tile by tile.
struct Image {
    int obj, blk, heads, head_tiles, prop_chunks, total;
    __host__ __device__ Image(int prop_dim, int layers, int n_out) {
        prop_chunks = (prop_dim + 31) / 32; head_tiles = (n_out + 15) / 16;
        obj = NT * prop_chunks; blk = obj + NT; heads = blk + layers * BLK_FRAGS; total = heads + head_tiles * KC;
    }
};
__global__ __launch_bounds__(256) void env_pack_kernel(bsrl_cfg_rows_weights w, uint4* img, int prop_dim, int obj_dim, int layers, int n_out) {
    const Image im(prop_dim, layers, n_out);
    const int f = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, g = lane >> 4;      // one wave per fragment
    if (f >= im.total) return;
    const void* src; int r, chunks = KC, K = D, rows = 1 << 30; bool pairs = false;
    if (f < im.obj) { src = w.prop_w; r = f; chunks = im.prop_chunks; K = prop_dim; }
    else if (f < im.blk) { src = w.obj_w; r = f - im.obj; chunks = 1; K = obj_dim; }
    else if (f >= im.heads) { src = w.heads_w; r = f - im.heads; rows = n_out; }
    else {
        const auto& k = w.blk[(f - im.blk) / BLK_FRAGS];
        r = (f - im.blk) % BLK_FRAGS;
        if (r < OUT_AT) src = k.qkv_w;
        else if (r < W0_AT) { src = k.out_w; r -= OUT_AT; pairs = true; }
        else if (r < W2_AT) { src = k.w0; r -= W0_AT; }
        else { src = k.w2; r -= W2_AT; chunks = F / 32; K = F; pairs = true; }
    }
    const int row = 16 * (r / chunks) + (lane & 15), c = r % chunks;
    u16 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int k = pairs ? bperm_k(c, g, j) : 32 * c + 8 * g + j;
        v[j] = row < rows && k < K ? static_cast<const u16*>(src)[(int64_t)row * K + k] : (u16)0;
    }
    uint4 o;
    o.x = v[0] | (uint32_t)v[1] << 16; o.y = v[2] | (uint32_t)v[3] << 16; o.z = v[4] | (uint32_t)v[5] << 16; o.w = v[6] | (uint32_t)v[7] << 16;
    img[(int64_t)f * 64 + lane] = o;
}

// A row dealt over 16 lanes, three 16-byte pieces (eight features) each: lane `sub` holds pieces sub + 16 i.
template <typename DT> __device__ __forceinline__ void unpack8(const uint4& u, float (&v)[8]) {
    const uint32_t q[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[2 * j] = DT::to_f((u16)(q[j] & 0xffff)); v[2 * j + 1] = DT::to_f((u16)(q[j] >> 16)); }
}
template <typename DT> __device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
    return make_uint4(DT::pack2(v[0], v[1]), DT::pack2(v[2], v[3]), DT::pack2(v[4], v[5]), DT::pack2(v[6], v[7]));
}
// a row's x1 and the four parts of what is added to it: x1 + b2 + the parts, rounded
struct RowParts {
    uint4 x1[3]; f32x4 p[3][2][SL];
    __device__ __forceinline__ void load(const u16* x, const float* part, int64_t pitch, int64_t row, int sub) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int64_t at = row * D + 8 * (sub + 16 * i);
            x1[i] = *reinterpret_cast<const uint4*>(x + at);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int k = 0; k < SL; ++k) p[i][h][k] = *reinterpret_cast<const f32x4*>(part + k * pitch + at + 4 * h);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    template <typename DT> __device__ __forceinline__ void sum(const float* b2, int sub, uint4 (&x)[3]) const {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            float v[8];
            unpack8<DT>(x1[i], v);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4 b = *reinterpret_cast<const f32x4*>(b2 + 8 * (sub + 16 * i) + 4 * h), t = (p[i][h][0] + p[i][h][1]) + (p[i][h][2] + p[i][h][3]);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * h + j] += t[j] + b[j];
            }
            x[i] = pack8<DT>(v);
        }
    }
};
// LayerNorm of the row (two passes, as ln_kernel) -> its places in the operand fragments [row tile][chunk][lane]; on: the row exists
template <typename DT> __device__ __forceinline__ void norm_row(const uint4 (&x)[3], const float* gamma, const float* beta, int row, int sub, bool on, uint4* hf) {
    float v[3][8], s = 0.f, q = 0.f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        unpack8<DT>(x[i], v[i]);
#pragma unroll
        for (int j = 0; j < 8; ++j) s += v[i][j];
    }
    const float mean = group_sum<16>(s) * (1.0f / D);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) { const float t = v[i][j] - mean; q = fmaf(t, t, q); }
    const float rstd = 1.0f / sqrtf(group_sum<16>(q) * (1.0f / D) + 1e-5f);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int p = sub + 16 * i;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 gm = *reinterpret_cast<const float4*>(gamma + 8 * p + 4 * h), bt = *reinterpret_cast<const float4*>(beta + 8 * p + 4 * h);
            v[i][4 * h] = (v[i][4 * h] - mean) * rstd * gm.x + bt.x; v[i][4 * h + 1] = (v[i][4 * h + 1] - mean) * rstd * gm.y + bt.y;
            v[i][4 * h + 2] = (v[i][4 * h + 2] - mean) * rstd * gm.z + bt.z; v[i][4 * h + 3] = (v[i][4 * h + 3] - mean) * rstd * gm.w + bt.w;
        }
        hf[((row >> 4) * KC + (p >> 2)) * 64 + 16 * (p & 3) + (row & 15)] = on ? pack8<DT>(v[i]) : make_uint4(0, 0, 0, 0);
    }
}
__device__ __forceinline__ s16x8 as_frag(const uint4& u) { return __builtin_bit_cast(s16x8, u); }

// One env's rows from a block's input to x1 = x + attention.  FIRST: the input comes from the tokenizer; FIN: the pruned final block.
struct BlockArgs {
    const uint4* img; const void* obs; int64_t obs_ld;
    const int32_t* noff; const u16* xin; u16* x1; const float* part; int64_t pitch;
    const float *prop_b, *obj_b, *b2, *ln_w, *ln_b, *qkv_b, *out_b;
    int prop_chunks, obj, blk, prop_dim, obj_dim, obs_f32, obs_vec;
};
constexpr int LNW = 0, LNB = D, VB2 = 2 * D, QKVB = 3 * D, OUTB = 6 * D, NVEC = 7 * D;        // the vectors in LDS
constexpr int BLOCK_LDS = 2 * 3 * KC * 64 * 16 + MT * XLD * 2 + NVEC * 4;

template <typename DT, bool FIRST, bool FIN>
__global__ __launch_bounds__(768, 3) void env_block_kernel(BlockArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint4 lds[];
    uint4* const hf = lds;                           // LayerNorm output [row tile][chunk][lane]
    uint4* const of = hf + 3 * KC * 64;              // attention's output, a head per chunk
    u16* const xs = reinterpret_cast<u16*>(of + 3 * KC * 64);        // the input rows
    float* const vec = reinterpret_cast<float*>(xs + MT * XLD);
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int b = blockIdx.x, o0 = a.noff[b], n = 1 + a.noff[b + 1] - o0;
    const int64_t row0 = (int64_t)b + o0;
    // weights: group k of four fragments (two chunks of two tiles), the wave's q (groups 0 - 5), k, v, output projection (18 - 23)
    uint4 wb[4][4];
    auto load = [&](auto k_) __attribute__((always_inline)) {
        constexpr int k = decltype(k_)::value, part = k / 6, c0 = 2 * (k % 6);
        const uint4* p = a.img + (int64_t)(a.blk + (part * NT + 2 * w) * KC) * 64 + lane;        // (the output projection follows v's tiles)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) wb[k % 4][i] = p[((i & 1) * KC + c0 + (i >> 1)) * 64];
        __builtin_amdgcn_sched_barrier(0);
    };
    typedef std::integral_constant<int, 0> G0; typedef std::integral_constant<int, 1> G1; typedef std::integral_constant<int, 2> G2; typedef std::integral_constant<int, 3> G3;
    // loads retire in order: what is wanted first goes first
    float4 v4 = make_float4(0.f, 0.f, 0.f, 0.f);
    if (tid < NVEC / 4) {
        const int at = 4 * tid;
        const float* p = at < LNB ? a.ln_w + at : at < VB2 ? a.ln_b + (at - LNB) : at < QKVB ? (FIRST ? a.ln_w : a.b2 + (at - VB2)) : at < OUTB ? a.qkv_b + (at - QKVB) : a.out_b + (at - OUTB);
        v4 = *reinterpret_cast<const float4*>(p);
    }
    load(G0());
    const int row = w + 12 * g, sub = r16;           // this lane's row in the row-wise parts
    uint4 x[3] = {};
    if constexpr (FIRST) {
        // tokens: K = proprio | object, feature tiles 2 w, 2 w + 1 of every row tile
        // eight observations from `at` + k on as an operand fragment, zero at and past K
        auto obs8 = [&](int64_t at, int k, int K, bool on) __attribute__((always_inline)) {
            float v[8];
            const int64_t i0 = (int64_t)b * a.obs_ld + at;
            if (a.obs_vec) {                         // fp32 rows on a 16-byte grid, K a multiple of four
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool in = on && k + 4 * h < K;
                    const float4 q = *reinterpret_cast<const float4*>(static_cast<const float*>(a.obs) + (in ? i0 + k + 4 * h : 0));
                    v[4 * h] = in ? q.x : 0.f; v[4 * h + 1] = in ? q.y : 0.f; v[4 * h + 2] = in ? q.z : 0.f; v[4 * h + 3] = in ? q.w : 0.f;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const bool in = on && k + j < K;
                    const int64_t i = in ? i0 + k + j : 0;
                    v[j] = a.obs_f32 ? static_cast<const float*>(a.obs)[i] : DT::to_f(static_cast<const u16*>(a.obs)[i]);
                    v[j] = in ? v[j] : 0.f;
                }
            }
            return as_frag(pack8<DT>(v));
        };
        auto tile_frag = [&](int at) __attribute__((always_inline)) { return as_frag(a.img[(int64_t)at * 64 + lane]); };
        f32x4 acc[2][3];
        s16x8 o[3], wo[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            wo[t] = tile_frag(a.obj + 2 * w + t);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int f = 16 * (2 * w + t) + 4 * g + i;
                const float bo = a.obj_b[f], bp = a.prop_b[f];
#pragma unroll
                for (int rt = 0; rt < 3; ++rt) acc[t][rt][i] = rt == 0 && r16 == 0 ? bp : bo;
            }
        }
#pragma unroll
        for (int rt = 0; rt < 3; ++rt) {
            const int r = 16 * rt + r16;
            o[rt] = obs8(a.prop_dim + (int64_t)(r - 1) * a.obj_dim, 8 * g, a.obj_dim, r >= 1 && r < n);
        }
        for (int c0 = 0; c0 < a.prop_chunks; c0 += 4) {
            s16x8 op[4], wp[2][4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                op[c] = obs8(0, 32 * (c0 + c) + 8 * g, a.prop_dim, r16 == 0);
#pragma unroll
                for (int t = 0; t < 2; ++t) wp[t][c] = tile_frag((2 * w + t) * a.prop_chunks + (c0 + c < a.prop_chunks ? c0 + c : 0));      // (times zeros past the end)
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int t = 0; t < 2; ++t) acc[t][0] = DT::mfma32(wp[t][c], op[c], acc[t][0]);
        }
#pragma unroll
        for (int rt = 0; rt < 3; ++rt)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                acc[t][rt] = DT::mfma32(wo[t], o[rt], acc[t][rt]);
                *reinterpret_cast<uint2*>(xs + (16 * rt + r16) * XLD + 16 * (2 * w + t) + 4 * g) =
                    make_uint2(DT::pack2(acc[t][rt][0], acc[t][rt][1]), DT::pack2(acc[t][rt][2], acc[t][rt][3]));
            }
        load(G1()); load(G2()); load(G3());
        if (tid < NVEC / 4) *reinterpret_cast<float4*>(vec + 4 * tid) = v4;
        blk_barrier();
#pragma unroll
        for (int i = 0; i < 3; ++i) x[i] = *reinterpret_cast<const uint4*>(xs + row * XLD + 8 * (sub + 16 * i));
    } else {
        RowParts parts;
        if (row < n) parts.load(a.xin, a.part, a.pitch, row0 + row, sub);
        if (tid < NVEC / 4) *reinterpret_cast<float4*>(vec + 4 * tid) = v4;
        blk_barrier();
        if (row < n) parts.sum<DT>(vec + VB2, sub, x);
        load(G1()); load(G2()); load(G3());
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(xs + row * XLD + 8 * (sub + 16 * i)) = x[i];
    }
    norm_row<DT>(x, vec + LNW, vec + LNB, row, sub, row < n, hf);
    blk_barrier();

    // nt: row tiles that hold rows (uniform branches around the others: three bodies of straight-line code would each come cold)
    const int nt = (n + 15) >> 4, nqt = FIN ? 1 : nt;
    constexpr int RT = 3, QT = FIN ? 1 : RT;
    BFrag8 qf[QT], kf[RT], vf[2][2];                 // V^T of two key tiles side by side
#pragma unroll
    for (int t = 0; t < 2; ++t) vf[t][0].u = vf[t][1].u = make_uint4(0, 0, 0, 0);
    static_for<0, 3>([&](auto p_) __attribute__((always_inline)) {
        constexpr int p = decltype(p_)::value, PT = p == 0 ? QT : RT;
        f32x4 acc[2][PT];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x4 bias;
            if constexpr (p < 2) bias = *reinterpret_cast<const f32x4*>(vec + QKVB + D * p + 32 * w + 16 * t + 4 * g);
            else { const float v = vec[QKVB + 2 * D + 32 * w + 16 * t + r16]; bias = (f32x4){v, v, v, v}; }
#pragma unroll
            for (int rt = 0; rt < PT; ++rt) acc[t][rt] = bias;
        }
        static_for<0, 6>([&](auto s_) __attribute__((always_inline)) {
            constexpr int s = decltype(s_)::value, k = 6 * p + s;
#pragma unroll
            for (int rt = 0; rt < PT; ++rt)
                if (rt == 0 || rt < nt) {
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        const s16x8 h = as_frag(hf[(rt * KC + 2 * s + c) * 64 + lane]);
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            const s16x8 wf = as_frag(wb[k % 4][2 * c + t]);
                            if constexpr (p < 2) acc[t][rt] = DT::mfma32(wf, h, acc[t][rt]);
                            else acc[t][rt] = DT::mfma32(h, wf, acc[t][rt]);       // V over keys: operand roles swapped
                        }
                    }
                }
            load(std::integral_constant<int, k + 4>());
        });
#pragma unroll
        for (int rt = 0; rt < PT; ++rt)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint2 v = make_uint2(DT::pack2(acc[t][rt][0], acc[t][rt][1]), DT::pack2(acc[t][rt][2], acc[t][rt][3]));
                if constexpr (p == 0) qf[rt].h[t] = v;
                else if constexpr (p == 1) kf[rt].h[t] = v;
                else if (rt == 0 || rt < nt) vf[t][rt >> 1].h[rt & 1] = v;         // (tiles past the rows stay zero: their probabilities are)
            }
    });
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {                // attention of head w: keys 16 kt + 4 g + i of query r16 in a lane
        if (qt > 0 && qt >= nqt) break;
        f32x4 s[RT];
        float m = -INFINITY, sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < RT; ++kt) {
            s[kt] = (f32x4){0.f, 0.f, 0.f, 0.f};
            if (kt > 0 && kt >= nt) { s[kt] = (f32x4){-INFINITY, -INFINITY, -INFINITY, -INFINITY}; continue; }
            s[kt] = DT::mfma32(kf[kt].v, qf[qt].v, s[kt]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[kt][i] = 16 * kt + 4 * g + i < n ? s[kt][i] * 0.17677669529663688110f : -INFINITY;
                m = fmaxf(m, s[kt][i]);
            }
        }
        float m1 = m;
        rows_reduce2(m, m1, OpMax());
#pragma unroll
        for (int kt = 0; kt < RT; ++kt) {
            if (kt > 0 && kt >= nt) { s[kt] = (f32x4){0.f, 0.f, 0.f, 0.f}; continue; }
#pragma unroll
            for (int i = 0; i < 4; ++i) { s[kt][i] = __expf(s[kt][i] - m); sum += s[kt][i]; }
        }
        float s1 = sum;
        rows_reduce2(sum, s1, OpAdd());
        const float inv = 1.0f / sum;
        BFrag8 pf[2];
        pf[1].u = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int kt = 0; kt < RT; ++kt) pf[kt >> 1].h[kt & 1] = make_uint2(DT::pack2(s[kt][0] * inv, s[kt][1] * inv), DT::pack2(s[kt][2] * inv, s[kt][3] * inv));
        BFrag8 o;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < 2; ++k) v = DT::mfma32(vf[t][k].v, pf[k].v, v);
            o.h[t] = make_uint2(DT::pack2(v[0], v[1]), DT::pack2(v[2], v[3]));
        }
        of[(qt * KC + w) * 64 + lane] = o.u;
    }
    blk_barrier();
    f32x4 acc[2][QT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int rt = 0; rt < QT; ++rt) acc[t][rt] = *reinterpret_cast<const f32x4*>(vec + OUTB + 32 * w + 16 * t + 4 * g);
    static_for<0, 6>([&](auto s_) __attribute__((always_inline)) {
        constexpr int s = decltype(s_)::value, k = 18 + s;
#pragma unroll
        for (int rt = 0; rt < QT; ++rt)
            if (rt == 0 || rt < nqt) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const s16x8 h = as_frag(of[(rt * KC + 2 * s + c) * 64 + lane]);
#pragma unroll
                    for (int t = 0; t < 2; ++t) acc[t][rt] = DT::mfma32(as_frag(wb[k % 4][2 * c + t]), h, acc[t][rt]);
                }
            }
        if constexpr (k + 4 < 24) load(std::integral_constant<int, k + 4>());
    });
#pragma unroll
    for (int rt = 0; rt < QT; ++rt) {
        const int r = 16 * rt + r16;
        if (r < (FIN ? 1 : n)) {
            u16* out = a.x1 + (FIN ? (int64_t)b : row0 + r) * D + 32 * w + 4 * g;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint2 v = *reinterpret_cast<const uint2*>(xs + r * XLD + 32 * w + 16 * t + 4 * g);
                uint2 y;
                y.x = DT::pack2(DT::to_f((u16)(v.x & 0xffff)) + acc[t][rt][0], DT::to_f((u16)(v.x >> 16)) + acc[t][rt][1]);
                y.y = DT::pack2(DT::to_f((u16)(v.y & 0xffff)) + acc[t][rt][2], DT::to_f((u16)(v.y >> 16)) + acc[t][rt][3]);
                *reinterpret_cast<uint2*>(out + 16 * t) = y;
            }
        }
    }
}

// part[s] of rows 32 t .. 32 t + 31 = the hidden's slice s through the down-projection; workgroup 4 t + s (an XCD then streams one slice)
struct FfnArgs {
    const uint4* img; const int32_t* extra; const u16* x1; float* part; int64_t pitch;
    const float *ln_w, *ln_b, *b0;
    int blk, rows;
};
template <typename DT, int ACT>
__global__ __launch_bounds__(512, 2) void env_ffn_kernel(FfnArgs a) {
    constexpr int ST = F / 16 / SL, PW = ST / 8;     // hidden tiles of a slice, tiles per wave (up and down)
    static_assert(ST == NT && PW == 3, "a wave has three tiles of either projection");
    __shared__ uint4 hf[2 * KC * 64], hid[2 * KC * 64];
    __shared__ __attribute__((aligned(16))) float vec[3 * D];        // LayerNorm, the slice's hidden biases
    const int tid = threadIdx.x;
    const int rows = a.rows + (a.extra ? *a.extra : 0), t0 = 32 * (int)(blockIdx.x / SL), sl = blockIdx.x % SL;
    if (t0 >= rows) return;
    const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    uint4 wb[PW][KC];
    auto load = [&](uint4 (&f)[KC], int at) __attribute__((always_inline)) {
        const uint4* p = a.img + (int64_t)(a.blk + at) * 64 + lane;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < KC; ++c) f[c] = p[c * 64];
        __builtin_amdgcn_sched_barrier(0);
    };
    // loads retire in order: what is wanted first goes first
    const int row = 4 * w + g, ar = t0 + row < rows ? t0 + row : rows - 1;
    uint4 x[3];
    float4 v4 = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < 3; ++i) x[i] = *reinterpret_cast<const uint4*>(a.x1 + (int64_t)ar * D + 8 * (r16 + 16 * i));
    if (tid < 3 * D / 4) v4 = *reinterpret_cast<const float4*>(tid < D / 4 ? a.ln_w + 4 * tid : tid < D / 2 ? a.ln_b + 4 * tid - D : a.b0 + D * sl + 4 * tid - 2 * D);
#pragma unroll
    for (int i = 0; i < PW; ++i) load(wb[i], W0_AT + (ST * sl + PW * w + i) * KC);
    if (tid < 3 * D / 4) *reinterpret_cast<float4*>(vec + 4 * tid) = v4;
    blk_barrier();
    norm_row<DT>(x, vec, vec + D, row, r16, true, hf);
    blk_barrier();
    f32x4 acc[2];
    auto run = [&](const uint4 (&f)[KC], const uint4* act) __attribute__((always_inline)) {
        acc[0] = acc[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) acc[rt] = DT::mfma32(as_frag(f[c]), as_frag(act[(rt * KC + c) * 64 + lane]), acc[rt]);
    };
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int lt = PW * w + i;
        const f32x4 b0 = *reinterpret_cast<const f32x4*>(vec + 2 * D + 16 * lt + 4 * g);
        run(wb[i], hf);
        load(wb[i], W2_AT + lt * (F / 32) + KC * sl);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const f32x4 v = acc[rt] + b0;
            reinterpret_cast<uint2*>(hid)[((rt * KC + (lt >> 1)) * 64 + lane) * 2 + (lt & 1)] =
                make_uint2(DT::pack2(apply_act16<ACT>(v[0]), apply_act16<ACT>(v[1])), DT::pack2(apply_act16<ACT>(v[2]), apply_act16<ACT>(v[3])));
        }
    }
    blk_barrier();
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        run(wb[i], hid);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const int r = t0 + 16 * rt + r16;
            if (r < rows) *reinterpret_cast<f32x4*>(a.part + sl * a.pitch + (int64_t)r * D + 16 * (PW * w + i) + 4 * g) = acc[rt];
        }
    }
}

// 32 envs' token 0 -> 29 K logits + value
struct HeadArgs {
    const uint4* img; const u16* x1; const float* part; int64_t pitch;
    const float *b2, *ln_w, *ln_b, *heads_b; float *logits, *value;
    int heads, head_tiles, n_out, B;
};
template <typename DT>
__global__ __launch_bounds__(512, 2) void env_heads_kernel(HeadArgs a) {
    __shared__ uint4 hf[2 * KC * 64];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int row = 4 * w + g, t0 = 32 * blockIdx.x, b = t0 + row < a.B ? t0 + row : a.B - 1;
    uint4 wf[KC], x[3];
    const int tile0 = w < a.head_tiles ? w : 0;
    RowParts parts;
    parts.load(a.x1, a.part, a.pitch, b, r16);
#pragma unroll
    for (int c = 0; c < KC; ++c) wf[c] = a.img[(int64_t)(a.heads + tile0 * KC + c) * 64 + lane];
    parts.sum<DT>(a.b2, r16, x);
    if (a.ln_w) norm_row<DT>(x, a.ln_w, a.ln_b, row, r16, true, hf);
    else {
#pragma unroll
        for (int i = 0; i < 3; ++i) { const int p = r16 + 16 * i; hf[((row >> 4) * KC + (p >> 2)) * 64 + 16 * (p & 3) + (row & 15)] = x[i]; }
    }
    blk_barrier();
    for (int t = w; t < a.head_tiles; t += 8) {
        if (t != w)
#pragma unroll
            for (int c = 0; c < KC; ++c) wf[c] = a.img[(int64_t)(a.heads + t * KC + c) * 64 + lane];
        f32x4 acc[2] = {};
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) acc[rt] = DT::mfma32(as_frag(wf[c]), as_frag(hf[(rt * KC + c) * 64 + lane]), acc[rt]);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const int e = t0 + 16 * rt + r16;
            if (e >= a.B) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = 16 * t + 4 * g + i;
                if (col + 1 < a.n_out) a.logits[(int64_t)e * (a.n_out - 1) + col] = acc[rt][i] + a.heads_b[col];
                else if (col + 1 == a.n_out) a.value[e] = acc[rt][i] + a.heads_b[col];
            }
        }
    }
}

template <typename DT, bool FIRST, bool FIN>
bool launch_block(const BlockArgs& a, int B, hipStream_t st) {
    auto kern = env_block_kernel<DT, FIRST, FIN>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, BLOCK_LDS) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)B), dim3(768), BLOCK_LDS, st, a);
    return true;
}

template <typename DT>
int forward(const bsrl_cfg_desc* d, const CfgEnvRowsArgs& a, hipStream_t st) {
    const int L = a.n_layers, B = a.B;
    const Image im(a.prop_dim, L, a.n_out);
    const uint4* img = static_cast<const uint4*>(a.w.lead_img);
    const int64_t pitch = (int64_t)B * a.T * D;
    for (int l = 0; l < L; ++l) {
        const auto& k = a.w.blk[l];
        const bool first = l == 0, fin = l + 1 == L;
        const int blk = im.blk + l * BLK_FRAGS;
        // (each env's x1 rows are read and written by its own workgroup alone, except behind the final block, whose row b is another
        // env's: there they go behind the last part's rows)
        u16* const x1 = fin ? a.x1 + pitch : a.x1;
        const BlockArgs p{img, a.obs, a.obs_ld, a.noff, a.x1, x1, a.part, pitch, a.w.prop_b, a.w.obj_b, first ? nullptr : a.w.blk[l - 1].b2, k.ln_attn_w, k.ln_attn_b,
                          k.qkv_b, k.out_b, im.prop_chunks, im.obj, blk, a.prop_dim, a.obj_dim, a.obs_f32,
                          a.obs_f32 && a.obs_ld % 4 == 0 && a.prop_dim % 4 == 0 && a.obj_dim % 4 == 0 && bsrl_aligned(a.obs, 16)};
        const bool ok = first ? (fin ? launch_block<DT, true, true>(p, B, st) : launch_block<DT, true, false>(p, B, st))
                              : (fin ? launch_block<DT, false, true>(p, B, st) : launch_block<DT, false, false>(p, B, st));
        if (!ok) return BSRL_UNSUPPORTED;
        const FfnArgs f{img, fin ? nullptr : a.noff + B, x1, a.part, pitch, k.ln_ffn_w, k.ln_ffn_b, k.b0, blk, B};
        const dim3 grid((unsigned)(((fin ? B : (int64_t)B * a.T) + 31) / 32 * SL));
        if (d->act == BSRL_ACT_GELU) hipLaunchKernelGGL((env_ffn_kernel<DT, BSRL_ACT_GELU>), grid, dim3(512), 0, st, f);
        else hipLaunchKernelGGL((env_ffn_kernel<DT, BSRL_ACT_RELU>), grid, dim3(512), 0, st, f);
    }
    const HeadArgs h{img, a.x1 + pitch, a.part, pitch, a.w.blk[L - 1].b2, a.final_ln ? a.w.final_ln_w : nullptr, a.w.final_ln_b, a.w.heads_b, a.logits, a.value,
                     im.heads, im.head_tiles, a.n_out, B};
    hipLaunchKernelGGL(env_heads_kernel<DT>, dim3((unsigned)((B + 31) / 32)), dim3(512), 0, st, h);
    BSRL_CHECK_LAUNCH("bsrl_cfg_rows_forward");
    return BSRL_OK;
}

}  // namespace

int64_t bsrl_cfg_env_rows_pack_size(const bsrl_cfg_desc* d) {
    if ((d->dtype != BSRL_F16 && d->dtype != BSRL_BF16) || d->d != D || d->n_heads != H || d->ffn != F || d->T > MT || d->prop_dim > 4096 || d->obj_dim > 32 ||
        d->n_gears > 64) return 0;
    return (int64_t)Image(d->prop_dim, d->n_layers, 29 * d->n_gears + 1).total * 1024;
}
int bsrl_cfg_env_rows_pack(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w, void* img, hipStream_t st) {
    const int n_out = 29 * d->n_gears + 1, total = Image(d->prop_dim, d->n_layers, n_out).total;
    hipLaunchKernelGGL(env_pack_kernel, dim3((unsigned)((total + 3) / 4)), dim3(256), 0, st, *w, static_cast<uint4*>(img), d->prop_dim, d->obj_dim, d->n_layers, n_out);
    BSRL_CHECK_LAUNCH("bsrl_cfg_rows_pack");
    return BSRL_OK;
}
bool bsrl_cfg_env_rows_ok(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w) {      // vectors in 16-byte pieces
    if (!w->lead_img || !bsrl_aligned(w->lead_img, 16) || bsrl_cfg_env_rows_pack_size(d) == 0) return false;
    bool ok = !d->final_ln || (bsrl_aligned(w->final_ln_w, 16) && bsrl_aligned(w->final_ln_b, 16));
    for (int l = 0; l < d->n_layers; ++l) {
        const auto& k = w->blk[l];
        for (const float* p : {k.ln_attn_w, k.ln_attn_b, k.ln_ffn_w, k.ln_ffn_b, k.qkv_b, k.out_b, k.b0, k.b2}) ok = ok && bsrl_aligned(p, 16);
    }
    return ok;
}
int bsrl_cfg_env_rows(const bsrl_cfg_desc* d, const CfgEnvRowsArgs& a, hipStream_t st) { return d->dtype == BSRL_F16 ? forward<F16>(d, a, st) : forward<BF16>(d, a, st); }
