// The transformer block stack of the policy in ONE persistent kernel for gfx950.
//
// Shape class: up to 32 tokens per env (NotePolicy: 29), d = 128 / 192 / 256 as 4 x 32, 4 x 48 or
// 8 x 32 heads, FFN width a multiple of 32, ReLU or GELU, fp16 or bf16 operands with fp32 accumulate.
// Replaces, for the block stack of NotePolicy._forward_stacked (python/policy.py:1262-1306),
// the per-block launch train of Block.forward (python/policy.py:524-715): LayerNorm, packed
// q|k|v projection, attention, output projection + residual, LayerNorm, FFN + residual,
// with the final block restricted to its first n_queries rows (the reference's n_queries
// path, python/policy.py:533-539: exact, masking is key-side only).
//
// Mapping.  One wave64 owns one 16-row MFMA tile of one env (rows 16*rt .. 16*rt + 15) and
// carries that tile's fp32 residual stream in registers through every block (d/16 feature
// tiles x 4 VGPRs).  An env is a wave pair; a workgroup of 8 waves owns 4 envs.  Everything
// row-local (LayerNorm, projections, FFN with the hidden kept in registers) is wave-local,
// with the activation always the MFMA operand whose free index is the token, so an output
// fragment (4 consecutive features per lane) packs straight into the next GEMM's operand;
// the k order this implies is baked into the weight image.  Only attention crosses the two
// row tiles: each wave parks its K and V^T fragments of the current head in LDS, and after
// the next stage barrier reads both tiles' fragments back (scores^T = K Q^T, 8 keys per
// lane for one query; softmax by in-lane + two cross-lane steps; P V as 16x16x32 MFMAs
// over the 32 keys).
//
// What bounds it: every weight fragment (1 KB) read from LDS feeds ONE MFMA of the reading wave,
// so a CU asks its LDS for 4 x 1 KB per 16 cycles = 256 B/clk against 128 B/clk delivered
// (measured): the stack runs at the LDS read rate, ~750 cycles per 12 KB stage.  Giving a wave both
// row tiles of an env halves that traffic but needs ~450 registers, i.e. one wave per SIMD; built
// and measured (3-slot ring, fragment reads prefetched across the barrier), it came out level at
// d = 128 and slower at d = 192 (register spills), each stage then waiting on the L2 latency of the
// weight stream (~1500 cycles) with no second wave to cover it.
//
// Weights stream from L2 through a 2-slot LDS ring in stages of 2 * (d/32) fragments
// (8 or 12 KB) shared by the 8 waves: loads issued three stages ahead into registers,
// written to LDS one stage ahead, one barrier per stage.  All fp32 vectors (biases,
// LayerNorm affine) of all blocks stay resident in LDS.  HBM traffic is the token stream in
// and the stream(s) out.
#include "block_stage.h"
#include "blocks_latency.h"
#include "blocks_pair.h"

namespace {

struct BlkArgs {
    const uint2* frags; const float* vec;
    const u16* x_in; const u16* key_bias; u16* x_res; u16* x_out;
    int64_t B; int n_layers, F, T, n_queries, total_stages;
    int per;                                  // blocks_env_kernel: envs per workgroup, 1 .. 8
    BlocksPairPlan plan;                      // d = 192, tiles not null: nothing to do where pairs pay (blocks_pair.hip)
};

// Weight-stage pipeline: stage s lives in ring slot s & 1; its global loads were issued three
// stage-steps earlier into the register set of the same parity.  The registers are plain named
// locals (an indexed array would live in scratch and force a wait right after each load).
#define BADVANCE_P(P, RA, RB, RC, RD) do { \
        blk_barrier();                                   /* stage s complete in slot P; slot 1-P free */ \
        ring[1 - (P)][tid] = RA; \
        ring[1 - (P)][tid + 512] = RB; \
        if (G::U2PT >= 3) ring[1 - (P)][tid + 1024] = RC; \
        if (G::U2PT == 4) ring[1 - (P)][tid + 1536] = RD; \
        const uint2* src_ = img + (int64_t)pnext * G::STAGE_U2 + tid; \
        RA = src_[0]; \
        RB = src_[512]; \
        if (G::U2PT >= 3) RC = src_[1024]; \
        if (G::U2PT == 4) RD = src_[1536]; \
        pnext = pnext + 1 == a.total_stages ? 0 : pnext + 1; \
    } while (0)
#define BADVANCE(par) do { if (par) BADVANCE_P(1, pr0a, pr0b, pr0c, pr0d); else BADVANCE_P(0, pr1a, pr1b, pr1c, pr1d); } while (0)
#define BWFRAG(par, f) (__builtin_bit_cast(s16x8, reinterpret_cast<const uint4*>(ring[par])[(f) * 64 + lane]))
// every fragment of the current stage -> registers in one burst of LDS reads (one wait instead of one per MFMA)
// one burst of a stage (FB fragments) -> registers in one run of LDS reads (one wait instead of one per MFMA).
// BLOAD_BURST: burst b of a two-tile stage, W[ntl * KB + ci] = k chunk b * KB + ci of tile ntl;
// BLOAD_RANGE: fragments [first, first + FB).
#define BLOAD_BURST(par, W, b) s16x8 W[G::FB]; _Pragma("unroll") for (int f_ = 0; f_ < G::FB; ++f_) W[f_] = BWFRAG(par, (b) * G::FB + f_)
#define BLOAD_RANGE(par, W, first) s16x8 W[G::FB]; _Pragma("unroll") for (int f_ = 0; f_ < G::FB; ++f_) W[f_] = BWFRAG(par, (first) + f_)

template <typename DT, int D, int DH, int ACT>
__global__ __launch_bounds__(512) void blocks_kernel(BlkArgs a) {
    typedef Geo<D> G;
    constexpr int NT = G::NT, KC = G::KC, H = D / DH, TPH = DH / 16;     // TPH: 16-feature tiles per head (2 or 3)
    constexpr int NB = G::NB, KB = G::KB, FB = G::FB;
    __shared__ __align__(16) uint2 ring[2][G::STAGE_U2];
    __shared__ uint2 kx[4][2][TPH][64];       // [env][row tile][feature tile of the head][lane]: K fragments
    __shared__ uint2 vx[4][2][TPH][64];       // V^T half fragments (this row tile's 4 keys per lane)
    extern __shared__ float4 bvl4[];          // fp32 vectors of every block
    const float* vlds = reinterpret_cast<const float*>(bvl4);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);     // in an SGPR: branches on it are scalar
    const int r16 = lane & 15, g = lane >> 4;
    const int el = wave >> 1, rt = wave & 1;
    const float scale_l2e = (DH == 32 ? 0.17677669529663688110f : 0.14433756729740644113f) * 1.44269504088896340736f;
    if (D == 192 && a.plan.tiles && blocks_pairs_pay(a.plan, blocks_pair_tiles(a.plan, lane))) return;
    const int64_t ntiles = (a.B + 3) / 4;

    const uint2* img = a.frags;
    const uint2 z2 = make_uint2(0, 0);
    uint2 pr0a, pr0b, pr0c = z2, pr0d = z2, pr1a, pr1b, pr1c = z2, pr1d = z2;
    int pnext;
    {   // prologue: stage 0 -> ring slot 0; stages 1 and 2 in flight (every block has an even stage count >= 4)
#pragma unroll
        for (int u = 0; u < G::U2PT; ++u) ring[0][tid + 512 * u] = img[tid + 512 * u];
        pr1a = img[G::STAGE_U2 + tid]; pr1b = img[G::STAGE_U2 + tid + 512];
        if (G::U2PT >= 3) pr1c = img[G::STAGE_U2 + tid + 1024];
        if (G::U2PT == 4) pr1d = img[G::STAGE_U2 + tid + 1536];
        pr0a = img[2 * G::STAGE_U2 + tid]; pr0b = img[2 * G::STAGE_U2 + tid + 512];
        if (G::U2PT >= 3) pr0c = img[2 * G::STAGE_U2 + tid + 1024];
        if (G::U2PT == 4) pr0d = img[2 * G::STAGE_U2 + tid + 1536];
        pnext = 3 % a.total_stages;
        const int nv4 = a.n_layers * G::lv_size(a.F) / 4;
        for (int i = tid; i < nv4; i += 512) bvl4[i] = reinterpret_cast<const float4*>(a.vec)[i];
        blk_barrier();
    }

    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t env = tile * 4 + el;
        const int64_t envc = env < a.B ? env : a.B - 1;
        const int row = 16 * rt + r16;
        const bool row_ok = row < a.T;
        f32x4 x[NT];
        BFrag8 hf[KC];       // LayerNorm output as operand fragments
        BFrag8 of[KC];       // attention output fragments
        float kmask[2][4];   // additive key bias * log2(e) for keys 16*kt + 4g + i; -inf past T
        {
            const u16* xr = a.x_in + (envc * a.T + (row_ok ? row : 0)) * D;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const uint2 v = *reinterpret_cast<const uint2*>(xr + 16 * nt + 4 * g);
                x[nt][0] = row_ok ? DT::to_f((u16)(v.x & 0xffff)) : 0.f;
                x[nt][1] = row_ok ? DT::to_f((u16)(v.x >> 16)) : 0.f;
                x[nt][2] = row_ok ? DT::to_f((u16)(v.y & 0xffff)) : 0.f;
                x[nt][3] = row_ok ? DT::to_f((u16)(v.y >> 16)) : 0.f;
            }
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int key = 16 * kt + 4 * g + i;
                    kmask[kt][i] = key < a.T ? DT::to_f(a.key_bias[envc * a.T + key]) * 1.44269504088896340736f : -INFINITY;
                }
        }

        auto norm_to_frags = [&](const float* gptr, const float* bptr) __attribute__((always_inline)) {
            // one pass: var = E[x^2] - mean^2 clamped at 0 (python/beat_arena_env/csrc/layer_norm.cu:14-21)
            float s = 0.f, q = 0.f;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) { s += x[nt][i]; q = fmaf(x[nt][i], x[nt][i], q); }
            s += __shfl_xor(s, 16, WAVE); q += __shfl_xor(q, 16, WAVE);
            s += __shfl_xor(s, 32, WAVE); q += __shfl_xor(q, 32, WAVE);
            const float mean = s * (1.0f / D);
            const float rstd = rsqrtf(fmaxf(fmaf(-mean, mean, q * (1.0f / D)), 0.f) + 1e-5f);
            const float shift = -mean * rstd;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const float4 gm = *reinterpret_cast<const float4*>(gptr + 16 * nt + 4 * g);
                const float4 bt = *reinterpret_cast<const float4*>(bptr + 16 * nt + 4 * g);
                const float y0 = fmaf(fmaf(x[nt][0], rstd, shift), gm.x, bt.x);
                const float y1 = fmaf(fmaf(x[nt][1], rstd, shift), gm.y, bt.y);
                const float y2 = fmaf(fmaf(x[nt][2], rstd, shift), gm.z, bt.z);
                const float y3 = fmaf(fmaf(x[nt][3], rstd, shift), gm.w, bt.w);
                hf[nt >> 1].w[(nt & 1) * 2] = bpack2<DT>(y0, y1);
                hf[nt >> 1].w[(nt & 1) * 2 + 1] = bpack2<DT>(y2, y3);
            }
        };
        auto add_bias = [&](const float* bptr) __attribute__((always_inline)) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const float4 b = *reinterpret_cast<const float4*>(bptr + 16 * nt + 4 * g);
                x[nt][0] += b.x; x[nt][1] += b.y; x[nt][2] += b.z; x[nt][3] += b.w;
            }
        };
        auto store_rows = [&](u16* dst, int rows_per_env, int nrows_valid) __attribute__((always_inline)) {
            // this wave's rows < nrows_valid of its env, 4 consecutive features (8 bytes) per lane and tile
            if (env < a.B && row < nrows_valid) {
                u16* o = dst + (env * rows_per_env + row) * D;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    uint2 v;
                    v.x = bpack2<DT>(x[nt][0], x[nt][1]); v.y = bpack2<DT>(x[nt][2], x[nt][3]);
                    *reinterpret_cast<uint2*>(o + 16 * nt + 4 * g) = v;
                }
            }
        };

        // one block; in the pruned final block only row tile 0 carries queries.  `pruned` is a compile-time
        // constant so that the full blocks carry no branches around their MFMAs.
        auto layer = [&](int l, auto pruned_) __attribute__((always_inline)) {
            constexpr bool pruned = decltype(pruned_)::value;
            const float* lv = vlds + l * G::lv_size(a.F);
            const bool active = !pruned || rt == 0;          // wave-uniform
            if (pruned && a.x_res) store_rows(a.x_res, a.T, a.T);

            norm_to_frags(lv + G::LN1G, lv + G::LN1B);

            uint2 q[2][TPH];                                  // Q fragments, double-buffered by head parity

            // attention of head hd for this wave's 16 queries over the env's 32 key slots
            auto attention = [&](auto hd_) __attribute__((always_inline)) {
                constexpr int hd = decltype(hd_)::value;
                if (!active) return;
                f32x4 sc[2];
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    BFrag8 kf, qf;
                    kf.h[0] = kx[el][kt][0][lane]; kf.h[1] = kx[el][kt][1][lane];
                    qf.h[0] = q[hd & 1][0]; qf.h[1] = q[hd & 1][1];
                    sc[kt] = DT::mfma32(kf.v, qf.v, (f32x4){0.f, 0.f, 0.f, 0.f});
                    if (TPH == 3) {
                        // features 32..47: a K = 16 MFMA into its OWN accumulator (chaining it onto the
                        // 16x16x32 accumulator loses the first product on this hardware), summed on the VALU
                        BFrag4 k2, q2;
                        k2.h = kx[el][kt][TPH - 1][lane]; q2.h = q[hd & 1][TPH - 1];
                        const f32x4 s2 = DT::mfma16(k2.v, q2.v, (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                        for (int i = 0; i < 4; ++i) sc[kt][i] += s2[i];
                    }
                }
                float sv[2][4];
                float m = -INFINITY;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) { sv[kt][i] = fmaf(sc[kt][i], scale_l2e, kmask[kt][i]); m = fmaxf(m, sv[kt][i]); }
                m = fmaxf(m, __shfl_xor(m, 16, WAVE)); m = fmaxf(m, __shfl_xor(m, 32, WAVE));
                float sum = 0.f;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) { sv[kt][i] = __builtin_amdgcn_exp2f(sv[kt][i] - m); sum += sv[kt][i]; }
                sum += __shfl_xor(sum, 16, WAVE); sum += __shfl_xor(sum, 32, WAVE);
                const float inv = __builtin_amdgcn_rcpf(sum);
                BFrag8 pf;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    pf.w[2 * kt] = bpack2<DT>(sv[kt][0] * inv, sv[kt][1] * inv);
                    pf.w[2 * kt + 1] = bpack2<DT>(sv[kt][2] * inv, sv[kt][3] * inv);
                }
#pragma unroll
                for (int t = 0; t < TPH; ++t) {
                    BFrag8 vf;
                    vf.h[0] = vx[el][0][t][lane]; vf.h[1] = vx[el][1][t][lane];
                    const float4 bv = *reinterpret_cast<const float4*>(lv + G::BV + DH * hd + 16 * t + 4 * g);
                    const f32x4 o = DT::mfma32(vf.v, pf.v, (f32x4){bv.x, bv.y, bv.z, bv.w});
                    const int nt = hd * TPH + t;
                    of[nt >> 1].w[(nt & 1) * 2] = bpack2<DT>(o[0], o[1]);
                    of[nt >> 1].w[(nt & 1) * 2 + 1] = bpack2<DT>(o[2], o[3]);
                }
            };

            // ---- packed q|k|v projection: 3 * NT feature tiles in head-major order
            //      [q tiles | k tiles | v tiles] per head, two tiles per stage ----
            static_for<0, 3 * NT / 2>([&](auto st_) __attribute__((always_inline)) {
                constexpr int st = decltype(st_)::value;
                BADVANCE(st & 1);
                // a head whose last tile was computed in an earlier stage is complete in LDS after this barrier
                if constexpr (st > 0) {
                    constexpr int done = (2 * st) / (3 * TPH);        // heads complete before this stage's first tile
                    constexpr int done_prev = (2 * st - 2) / (3 * TPH);
                    if constexpr (done > done_prev) attention(std::integral_constant<int, done - 1>{});
                }
                f32x4 acc[2];
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl) {
                    const int j = 2 * st + ntl, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;
                    float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (part < 2) b = *reinterpret_cast<const float4*>(lv + (part == 0 ? G::BQ : G::BK) + DH * hd + 16 * t + 4 * g);
                    acc[ntl] = (f32x4){b.x, b.y, b.z, b.w};
                }
#pragma unroll
                for (int half = 0; half < NB; ++half) {
                    BLOAD_BURST(st & 1, wf, half);                     // k chunks [half * KB, +KB) of both tiles
#pragma unroll
                    for (int ci = 0; ci < KB; ++ci)
#pragma unroll
                        for (int ntl = 0; ntl < 2; ++ntl) {
                            const int c = half * KB + ci;
                            const int j = 2 * st + ntl, part = (j % (3 * TPH)) / TPH;
                            if (part == 0 && !active) continue;        // the pruned block needs no queries from row tile 1
                            const s16x8 w = wf[ntl * KB + ci];
                            if (part < 2) acc[ntl] = DT::mfma32(w, hf[c].v, acc[ntl]);
                            else acc[ntl] = DT::mfma32(hf[c].v, w, acc[ntl]);   // V^T: operand roles swapped
                        }
                }
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl) {
                    const int j = 2 * st + ntl, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;
                    uint2 pk;
                    pk.x = bpack2<DT>(acc[ntl][0], acc[ntl][1]); pk.y = bpack2<DT>(acc[ntl][2], acc[ntl][3]);
                    if (part == 0) q[hd & 1][t] = pk;
                    else if (part == 1) kx[el][rt][t][lane] = pk;
                    else vx[el][rt][t][lane] = pk;
                }
            });

            // ---- output projection onto the residual (NT / 2 stages) ----
            if (active) add_bias(lv + G::BOUT);
            static_for<0, NT / 2>([&](auto st_) __attribute__((always_inline)) {
                constexpr int st = decltype(st_)::value;
                BADVANCE((3 * NT / 2 + st) & 1);
                if constexpr (st == 0) attention(std::integral_constant<int, H - 1>{});               // the last head completed in the previous stage
#pragma unroll
                for (int half = 0; half < NB; ++half) {
                    if (active) {            // idle waves of the pruned block leave the LDS bandwidth to the others
                        BLOAD_BURST((3 * NT / 2 + st) & 1, wf, half);
#pragma unroll
                        for (int ci = 0; ci < KB; ++ci)
#pragma unroll
                            for (int ntl = 0; ntl < 2; ++ntl)
                                x[2 * st + ntl] = DT::mfma32(wf[ntl * KB + ci], of[half * KB + ci].v, x[2 * st + ntl]);
                    }
                }
            });

            // ---- LayerNorm + FFN: stage order W1(0), {W1(ch+1), W2(ch)}..., W2(last); the hidden of a
            //      32-unit chunk lives in two accumulators, activated and packed into one operand fragment ----
            constexpr int P0 = (3 * NT / 2 + NT / 2) & 1;              // stage parity at FFN entry (0: 2 * NT is even)
            static_assert(P0 == 0, "FFN stages start on an even stage");
            if (active) { norm_to_frags(lv + G::LN2G, lv + G::LN2B); add_bias(lv + G::b2(a.F)); }
            const int nch = a.F / 32;
            f32x4 accA[2];
            auto up = [&](int par, int ch, f32x4 (&acc)[2]) __attribute__((always_inline)) {
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl) {
                    const float4 b = *reinterpret_cast<const float4*>(lv + G::B1 + 32 * ch + 16 * ntl + 4 * g);
                    acc[ntl] = (f32x4){b.x, b.y, b.z, b.w};
                }
#pragma unroll
                for (int half = 0; half < NB; ++half) {
                    if (active) {
                        BLOAD_BURST(par, wf, half);
#pragma unroll
                        for (int ci = 0; ci < KB; ++ci)
#pragma unroll
                            for (int ntl = 0; ntl < 2; ++ntl)
                                acc[ntl] = DT::mfma32(wf[ntl * KB + ci], hf[half * KB + ci].v, acc[ntl]);
                    }
                }
            };
            BADVANCE(0);
            up(0, 0, accA);
            for (int ch = 0; ch < nch; ++ch) {
                BFrag8 hid;
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl) {
                    hid.w[ntl * 2] = bpack2<DT>(apply_act16<ACT>(accA[ntl][0]), apply_act16<ACT>(accA[ntl][1]));
                    hid.w[ntl * 2 + 1] = bpack2<DT>(apply_act16<ACT>(accA[ntl][2]), apply_act16<ACT>(accA[ntl][3]));
                }
                if (ch + 1 < nch) {
                    BADVANCE(1);
                    up(1, ch + 1, accA);
                    BADVANCE(0);
#pragma unroll
                    for (int half = 0; half < NB; ++half) {
                        if (active) {
                            BLOAD_RANGE(0, w2, half * FB);
#pragma unroll
                            for (int i = 0; i < FB; ++i) x[half * FB + i] = DT::mfma32(w2[i], hid.v, x[half * FB + i]);
                        }
                    }
                } else {
                    BADVANCE(1);
#pragma unroll
                    for (int half = 0; half < NB; ++half) {
                        if (active) {
                            BLOAD_RANGE(1, w2, half * FB);
#pragma unroll
                            for (int i = 0; i < FB; ++i) x[half * FB + i] = DT::mfma32(w2[i], hid.v, x[half * FB + i]);
                        }
                    }
                }
            }
        };
        const int n_full = a.n_queries > 0 ? a.n_layers - 1 : a.n_layers;
        for (int l = 0; l < n_full; ++l) layer(l, std::false_type{});
        if (a.n_queries > 0) layer(a.n_layers - 1, std::true_type{});
        if (a.n_queries > 0) { if (rt == 0) store_rows(a.x_out, a.n_queries, a.n_queries); }
        else store_rows(a.x_out, a.T, a.T);
    }
}



// ---- the same stack with ONE WAVE PER ENV ---------------------------------------------------------------------
// Mapping.  A wave owns both 16-row tiles of an env (all its <= 32 tokens) and carries their fp32 residual stream in
// registers; a workgroup is 8 waves = 8 envs, one workgroup per CU, two waves per SIMD in 256 registers each.
// Against blocks_kernel (a wave per row tile, an env a wave pair, 4 envs per workgroup):
//   * every weight fragment read from LDS feeds TWO MFMAs (one per row tile) instead of one, and a stage streamed from
//     L2 serves 8 envs instead of 4: half the LDS read instructions, barriers and stage loads per env;
//   * attention needs no LDS: a wave holds the K and V^T fragments of both key tiles of the head it just projected;
//   * stages go global -> LDS directly (global_load_lds_dwordx4, one 1 KB fragment per wave instruction) several
//     stages ahead into a ring of SLOTS stage slots: no register staging, depth bounded by LDS only;
//   * the row reductions of LayerNorm and softmax are lane-row swaps on the VALU, not shuffles through LDS.
// Per-row arithmetic, its order and the weight image are those of blocks_kernel: an env's output bits are the same.
template <int D> struct EnvRing : StageRing<Geo<D>::SF, D == 128 ? 10 : 7> {};

template <typename DT, int D, int DH, int ACT>
__global__ __launch_bounds__(512, 1) void blocks_env_kernel(BlkArgs a) {
    typedef Geo<D> G;
    typedef EnvRing<D> R;
    constexpr int NW = R::NW;
    constexpr int NT = G::NT, KC = G::KC, H = D / DH, TPH = DH / 16;
    constexpr int NB = G::NB, KB = G::KB, SF = G::SF;
    // a stage is consumed in 2 * NB sub-bursts of KB fragments (a burst of blocks_kernel is two of them: the k chunks
    // [b * KB, +KB) of the stage's first tile, then of its second; in a W2 stage KB consecutive feature tiles)
    constexpr int NSUB = 2 * NB;
    static_assert(G::FB == 2 * KB, "a burst is two sub-bursts");
    extern __shared__ float4 bvl4[];          // fp32 vectors of every block, then the stage ring (1 KB aligned)
    const float* vlds = reinterpret_cast<const float*>(bvl4);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const float scale_l2e = (DH == 32 ? 0.17677669529663688110f : 0.14433756729740644113f) * 1.44269504088896340736f;
    if (D == 192 && a.plan.tiles && blocks_pairs_pay(a.plan, blocks_pair_tiles(a.plan, lane))) return;
    const int64_t ntiles = (a.B + a.per - 1) / a.per;
    const int ring_off_u4 = (a.n_layers * G::lv_size(a.F) / 4 + 63) & ~63;
    const uint4* ring = reinterpret_cast<const uint4*>(bvl4) + ring_off_u4;
    R pipe;
    auto advance = [&](auto parity_) __attribute__((always_inline)) { pipe.template admit<decltype(parity_)::value>(); };
    typedef std::integral_constant<int, 0> Even;
    typedef std::integral_constant<int, 1> Odd;
    // sub-burst j of the current stage -> registers, then `body` on them
    auto sub = [&](auto j_, auto&& body) __attribute__((always_inline)) {
        constexpr int j = decltype(j_)::value;
        s16x8 w[KB];
#pragma unroll
        for (int f = 0; f < KB; ++f) w[f] = pipe.frag(j * KB + f, lane);
        body(w);
    };
    {   // prologue: SLOTS - 2 stages in flight (every stack has more), then the vectors
        pipe.start(ring, a.frags, a.total_stages, wave, lane);
        const int nv4 = a.n_layers * G::lv_size(a.F) / 4;
        for (int i = tid; i < nv4; i += NW * 64) bvl4[i] = reinterpret_cast<const float4*>(a.vec)[i];
        blk_barrier();
    }

    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t env = tile * a.per + wave;
        if (wave >= a.per || env >= a.B) {        // no env: this wave only moves its share of the weight stream
            for (int s = 0; s < a.total_stages; s += 2) { advance(Even{}); advance(Odd{}); }
            continue;
        }
        f32x4 x[2][NT];
        BFrag8 hf[2][KC];    // LayerNorm output as operand fragments
        BFrag8 of[2][KC];    // attention output fragments
        float kmask[2][4];   // additive key bias * log2(e) for keys 16*kt + 4g + i; -inf past T
        // the tile's own loads are all issued, then waited for ONCE, with the wait the compiler can see (vmcnt(0); expcnt /
        // lgkmcnt at their maxima).  It does not know of the ring's loads: wherever it later met a value of its own still
        // in flight - or reused such a register - it would wait for every outstanding load, i.e. drain the ring in mid-tile.
        uint2 raw[2][NT];
        u16 kraw[2][4];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const int row = 16 * rt + r16;
            const u16* xr = a.x_in + (env * a.T + (row < a.T ? row : 0)) * D;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) raw[rt][nt] = *reinterpret_cast<const uint2*>(xr + 16 * nt + 4 * g);
        }
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = 16 * kt + 4 * g + i;
                kraw[kt][i] = a.key_bias[env * a.T + (key < a.T ? key : 0)];
            }
        __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const bool row_ok = 16 * rt + r16 < a.T;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const uint32_t lo = row_ok ? raw[rt][nt].x : 0u, hi = row_ok ? raw[rt][nt].y : 0u;      // 0 bits = +0.0
                x[rt][nt][0] = DT::to_f((u16)(lo & 0xffff)); x[rt][nt][1] = DT::to_f((u16)(lo >> 16));
                x[rt][nt][2] = DT::to_f((u16)(hi & 0xffff)); x[rt][nt][3] = DT::to_f((u16)(hi >> 16));
            }
        }
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                kmask[kt][i] = 16 * kt + 4 * g + i < a.T ? DT::to_f(kraw[kt][i]) * 1.44269504088896340736f : -INFINITY;

        // LayerNorm of both row tiles (of row tile 0 only: `both` false) -> operand fragments; the statistics of the two
        // tiles go through the lane-row butterfly together
        auto norm_to_frags = [&](bool both, const float* gptr, const float* bptr) __attribute__((always_inline)) {
            // one pass: var = E[x^2] - mean^2 clamped at 0 (python/beat_arena_env/csrc/layer_norm.cu:14-21)
            float s[2] = {0.f, 0.f}, q[2] = {0.f, 0.f};
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                if (rt == 1 && !both) break;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) { s[rt] += x[rt][nt][i]; q[rt] = fmaf(x[rt][nt][i], x[rt][nt][i], q[rt]); }
            }
            rows_reduce2(s[0], q[0], OpAdd());
            if (both) rows_reduce2(s[1], q[1], OpAdd());
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                if (rt == 1 && !both) break;
                const float mean = s[rt] * (1.0f / D);
                const float rstd = rsqrtf(fmaxf(fmaf(-mean, mean, q[rt] * (1.0f / D)), 0.f) + 1e-5f);
                const float shift = -mean * rstd;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float4 gm = *reinterpret_cast<const float4*>(gptr + 16 * nt + 4 * g);
                    const float4 bt = *reinterpret_cast<const float4*>(bptr + 16 * nt + 4 * g);
                    const float y0 = fmaf(fmaf(x[rt][nt][0], rstd, shift), gm.x, bt.x);
                    const float y1 = fmaf(fmaf(x[rt][nt][1], rstd, shift), gm.y, bt.y);
                    const float y2 = fmaf(fmaf(x[rt][nt][2], rstd, shift), gm.z, bt.z);
                    const float y3 = fmaf(fmaf(x[rt][nt][3], rstd, shift), gm.w, bt.w);
                    hf[rt][nt >> 1].w[(nt & 1) * 2] = bpack2<DT>(y0, y1);
                    hf[rt][nt >> 1].w[(nt & 1) * 2 + 1] = bpack2<DT>(y2, y3);
                }
            }
        };
        auto add_bias = [&](auto rt_, const float* bptr) __attribute__((always_inline)) {
            constexpr int rt = decltype(rt_)::value;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const float4 b = *reinterpret_cast<const float4*>(bptr + 16 * nt + 4 * g);
                x[rt][nt][0] += b.x; x[rt][nt][1] += b.y; x[rt][nt][2] += b.z; x[rt][nt][3] += b.w;
            }
        };
        auto store_rows = [&](auto rt_, u16* dst, int rows_per_env, int nrows_valid) __attribute__((always_inline)) {
            constexpr int rt = decltype(rt_)::value;
            const int row = 16 * rt + r16;
            if (row < nrows_valid) {
                u16* o = dst + (env * rows_per_env + row) * D;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    uint2 v;
                    v.x = bpack2<DT>(x[rt][nt][0], x[rt][nt][1]); v.y = bpack2<DT>(x[rt][nt][2], x[rt][nt][3]);
                    *reinterpret_cast<uint2*>(o + 16 * nt + 4 * g) = v;
                }
            }
        };
        typedef std::integral_constant<int, 0> T0;
        typedef std::integral_constant<int, 1> T1;

        // one block; the pruned final block computes queries, output projection and FFN for row tile 0 only (keys and
        // values of both).  `pruned` is a compile-time constant: the full blocks carry no branches around their MFMAs.
        auto layer = [&](int l, auto pruned_) __attribute__((always_inline)) {
            constexpr bool pruned = decltype(pruned_)::value;
            constexpr int QT = pruned ? 1 : 2;                 // query row tiles
            const float* lv = vlds + l * G::lv_size(a.F);
            if (pruned && a.x_res) { store_rows(T0(), a.x_res, a.T, a.T); store_rows(T1(), a.x_res, a.T, a.T); }

            norm_to_frags(true, lv + G::LN1G, lv + G::LN1B);

            uint2 q[2][2][TPH];                                // Q fragments [head parity][row tile][feature tile]
            uint2 kk[2][TPH], vv[2][TPH];                      // K, V^T fragments of the head in flight [key tile][feature tile]

            // attention of head hd: the env's (up to) 32 queries over its 32 key slots, both query tiles together
            auto attention = [&](auto hd_) __attribute__((always_inline)) {
                constexpr int hd = decltype(hd_)::value;
                float sv[2][2][4], m[2], sum[2];
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    f32x4 sc[2];
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        BFrag8 kf, qf;
                        kf.h[0] = kk[kt][0]; kf.h[1] = kk[kt][1];
                        qf.h[0] = q[hd & 1][qt][0]; qf.h[1] = q[hd & 1][qt][1];
                        sc[kt] = DT::mfma32(kf.v, qf.v, (f32x4){0.f, 0.f, 0.f, 0.f});
                        if (TPH == 3) {
                            // features 32..47: a K = 16 MFMA into its OWN accumulator (chaining it onto the
                            // 16x16x32 accumulator loses the first product on this hardware), summed on the VALU
                            BFrag4 k2, q2;
                            k2.h = kk[kt][TPH - 1]; q2.h = q[hd & 1][qt][TPH - 1];
                            const f32x4 s2 = DT::mfma16(k2.v, q2.v, (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                            for (int i = 0; i < 4; ++i) sc[kt][i] += s2[i];
                        }
                    }
                    m[qt] = -INFINITY;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) { sv[qt][kt][i] = fmaf(sc[kt][i], scale_l2e, kmask[kt][i]); m[qt] = fmaxf(m[qt], sv[qt][kt][i]); }
                }
                if (QT == 1) m[1] = m[0];
                rows_reduce2(m[0], m[1], OpMax());
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    sum[qt] = 0.f;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) { sv[qt][kt][i] = __builtin_amdgcn_exp2f(sv[qt][kt][i] - m[qt]); sum[qt] += sv[qt][kt][i]; }
                }
                if (QT == 1) sum[1] = sum[0];
                rows_reduce2(sum[0], sum[1], OpAdd());
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    const float inv = __builtin_amdgcn_rcpf(sum[qt]);
                    BFrag8 pf;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        pf.w[2 * kt] = bpack2<DT>(sv[qt][kt][0] * inv, sv[qt][kt][1] * inv);
                        pf.w[2 * kt + 1] = bpack2<DT>(sv[qt][kt][2] * inv, sv[qt][kt][3] * inv);
                    }
#pragma unroll
                    for (int t = 0; t < TPH; ++t) {
                        BFrag8 vf;
                        vf.h[0] = vv[0][t]; vf.h[1] = vv[1][t];
                        const float4 bv = *reinterpret_cast<const float4*>(lv + G::BV + DH * hd + 16 * t + 4 * g);
                        const f32x4 o = DT::mfma32(vf.v, pf.v, (f32x4){bv.x, bv.y, bv.z, bv.w});
                        const int nt = hd * TPH + t;
                        of[qt][nt >> 1].w[(nt & 1) * 2] = bpack2<DT>(o[0], o[1]);
                        of[qt][nt >> 1].w[(nt & 1) * 2 + 1] = bpack2<DT>(o[2], o[3]);
                    }
                }
            };

            // ---- packed q|k|v projection: 3 * NT feature tiles in head-major order [q | k | v] per head, two per stage ----
            static_for<0, 3 * NT / 2>([&](auto st_) __attribute__((always_inline)) {
                constexpr int st = decltype(st_)::value;
                advance(std::integral_constant<int, st & 1>{});
                // a head whose last tile was computed in an earlier stage is complete now: its attention runs before
                // this stage's results overwrite the K / V registers (a stage that straddles two heads holds the LAST
                // tile of one and the FIRST - a query tile, double-buffered by head parity - of the next)
                if constexpr (st > 0) {
                    constexpr int done = (2 * st) / (3 * TPH);
                    constexpr int done_prev = (2 * st - 2) / (3 * TPH);
                    if constexpr (done > done_prev) attention(std::integral_constant<int, done - 1>{});
                }
                f32x4 acc[2][2];                                 // [tile of the stage][row tile]
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl) {
                    const int j = 2 * st + ntl, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;
                    float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (part < 2) b = *reinterpret_cast<const float4*>(lv + (part == 0 ? G::BQ : G::BK) + DH * hd + 16 * t + 4 * g);
                    acc[ntl][0] = (f32x4){b.x, b.y, b.z, b.w}; acc[ntl][1] = acc[ntl][0];
                }
                static_for<0, NSUB>([&](auto j_) __attribute__((always_inline)) {
                    constexpr int half = decltype(j_)::value / 2, ntl = decltype(j_)::value % 2;    // k chunks [half * KB, +KB) of tile ntl
                    sub(j_, [&](const s16x8 (&wf)[KB]) __attribute__((always_inline)) {
#pragma unroll
                        for (int ci = 0; ci < KB; ++ci)
#pragma unroll
                            for (int rt = 0; rt < 2; ++rt) {
                                const int c = half * KB + ci;
                                const int j = 2 * st + ntl, part = (j % (3 * TPH)) / TPH;
                                if (part == 0 && rt >= QT) continue;     // the pruned block needs no queries from row tile 1
                                if (part < 2) acc[ntl][rt] = DT::mfma32(wf[ci], hf[rt][c].v, acc[ntl][rt]);
                                else acc[ntl][rt] = DT::mfma32(hf[rt][c].v, wf[ci], acc[ntl][rt]);   // V^T: operand roles swapped
                            }
                    });
                });
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl)
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt) {
                        const int j = 2 * st + ntl, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;
                        if (part == 0 && rt >= QT) continue;
                        uint2 pk;
                        pk.x = bpack2<DT>(acc[ntl][rt][0], acc[ntl][rt][1]); pk.y = bpack2<DT>(acc[ntl][rt][2], acc[ntl][rt][3]);
                        if (part == 0) q[hd & 1][rt][t] = pk;
                        else if (part == 1) kk[rt][t] = pk;
                        else vv[rt][t] = pk;
                    }
            });

            // ---- output projection onto the residual (NT / 2 stages) ----
            add_bias(T0(), lv + G::BOUT);
            if (!pruned) add_bias(T1(), lv + G::BOUT);
            static_for<0, NT / 2>([&](auto st_) __attribute__((always_inline)) {
                constexpr int st = decltype(st_)::value;
                advance(std::integral_constant<int, st & 1>{});
                if constexpr (st == 0) attention(std::integral_constant<int, H - 1>{});      // the last head completed in the previous stage
                static_for<0, NSUB>([&](auto j_) __attribute__((always_inline)) {
                    constexpr int half = decltype(j_)::value / 2, ntl = decltype(j_)::value % 2;
                    sub(j_, [&](const s16x8 (&wf)[KB]) __attribute__((always_inline)) {
#pragma unroll
                        for (int ci = 0; ci < KB; ++ci)
#pragma unroll
                            for (int qt = 0; qt < QT; ++qt)
                                x[qt][2 * st + ntl] = DT::mfma32(wf[ci], of[qt][half * KB + ci].v, x[qt][2 * st + ntl]);
                    });
                });
            });

            // ---- LayerNorm + FFN: stage order W1(0), {W1(ch+1), W2(ch)}..., W2(last); the hidden of a 32-unit chunk
            //      lives in two accumulators per row tile, activated and packed into one operand fragment ----
            norm_to_frags(!pruned, lv + G::LN2G, lv + G::LN2B);
            add_bias(T0(), lv + G::b2(a.F));
            if (!pruned) add_bias(T1(), lv + G::b2(a.F));
            const int nch = a.F / 32;
            f32x4 acc[2][2];                                     // [tile of the chunk][row tile]
            auto up = [&](int ch) __attribute__((always_inline)) {
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl) {
                    const float4 b = *reinterpret_cast<const float4*>(lv + G::B1 + 32 * ch + 16 * ntl + 4 * g);
                    acc[ntl][0] = (f32x4){b.x, b.y, b.z, b.w}; acc[ntl][1] = acc[ntl][0];
                }
                static_for<0, NSUB>([&](auto j_) __attribute__((always_inline)) {
                    constexpr int half = decltype(j_)::value / 2, ntl = decltype(j_)::value % 2;
                    sub(j_, [&](const s16x8 (&wf)[KB]) __attribute__((always_inline)) {
#pragma unroll
                        for (int ci = 0; ci < KB; ++ci)
#pragma unroll
                            for (int qt = 0; qt < QT; ++qt)
                                acc[ntl][qt] = DT::mfma32(wf[ci], hf[qt][half * KB + ci].v, acc[ntl][qt]);
                    });
                });
            };
            static_assert((3 * NT / 2) % 2 == 0 && (NT / 2) % 2 == 0, "the FFN starts on an even stage");
            advance(Even{});
            up(0);
            for (int ch = 0; ch < nch; ++ch) {
                BFrag8 hid[2];
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                    for (int ntl = 0; ntl < 2; ++ntl) {
                        hid[qt].w[ntl * 2] = bpack2<DT>(apply_act16<ACT>(acc[ntl][qt][0]), apply_act16<ACT>(acc[ntl][qt][1]));
                        hid[qt].w[ntl * 2 + 1] = bpack2<DT>(apply_act16<ACT>(acc[ntl][qt][2]), apply_act16<ACT>(acc[ntl][qt][3]));
                    }
                // stage parities: W1(0) even, then {W1(ch + 1) odd, W2(ch) even} ..., W2(last) odd
                if (ch + 1 < nch) { advance(Odd{}); up(ch + 1); advance(Even{}); }
                else advance(Odd{});
                static_for<0, NSUB>([&](auto j_) __attribute__((always_inline)) {
                    constexpr int j = decltype(j_)::value;           // feature tiles [j * KB, +KB)
                    sub(j_, [&](const s16x8 (&w2)[KB]) __attribute__((always_inline)) {
#pragma unroll
                        for (int i = 0; i < KB; ++i)
#pragma unroll
                            for (int qt = 0; qt < QT; ++qt) x[qt][j * KB + i] = DT::mfma32(w2[i], hid[qt].v, x[qt][j * KB + i]);
                    });
                });
            }
        };
        const int n_full = a.n_queries > 0 ? a.n_layers - 1 : a.n_layers;
        for (int l = 0; l < n_full; ++l) layer(l, std::false_type{});
        if (a.n_queries > 0) layer(a.n_layers - 1, std::true_type{});
        if (a.n_queries > 0) store_rows(T0(), a.x_out, a.n_queries, a.n_queries);
        else { store_rows(T0(), a.x_out, a.T, a.T); store_rows(T1(), a.x_out, a.T, a.T); }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // no transfer into LDS may outlive the workgroup
    blk_barrier();
}

// ---- weight image ------------------------------------------------------------------
struct BlkPackArgs {
    bsrl_blocks_params p;
    void* frags; float* vec;
    int n_layers, F;
};

// one wave per fragment, one lane per 16-byte slot
template <typename DT, int D, int DH>
__global__ __launch_bounds__(256) void blocks_pack_frags_kernel(BlkPackArgs a) {
    typedef Geo<D> G;
    constexpr int NT = G::NT, KC = G::KC, SF = G::SF, TPH = DH / 16;
    const int lane = threadIdx.x & 63;
    const int lfr = G::layer_stages(a.F) * SF;                 // fragments per block
    const int f = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (f >= a.n_layers * lfr) return;
    const int n16 = lane & 15, gg = lane >> 4;
    const int l = f / lfr, r = f % lfr;
    const auto& b = a.p.blk[l];
    const float* src; int ld, n, kbase = 0, c;
    // inside a stage of two feature tiles the fragments are ordered (burst, tile, k chunk of the burst):
    // consecutive runs of FB fragments are what a consumer reads together
    auto split = [&](int i, int& ntl, int& cc) {
        const int burst = i / G::FB, rem = i % G::FB;
        ntl = rem / G::KB; cc = burst * G::KB + rem % G::KB;
    };
    if (r < 3 * NT * KC) {
        int ntl; split(r % SF, ntl, c);
        const int j = 2 * (r / SF) + ntl, hd = j / (3 * TPH), rr = j % (3 * TPH), part = rr / TPH, t = rr % TPH;
        src = part == 0 ? b.q_w : part == 1 ? b.k_w : b.v_w;
        ld = D; n = DH * hd + 16 * t + n16;
    } else if (r < 4 * NT * KC) {
        const int r2 = r - 3 * NT * KC;
        int ntl; split(r2 % SF, ntl, c);
        src = b.out_w; ld = D; n = 16 * (2 * (r2 / SF) + ntl) + n16;
    } else {
        const int r3 = r - 4 * NT * KC, s3 = r3 / SF, i = r3 % SF, nch = a.F / 32;
        bool upw; int ch;
        if (s3 == 0) { upw = true; ch = 0; }
        else if (s3 == 2 * nch - 1) { upw = false; ch = nch - 1; }
        else { upw = ((s3 - 1) & 1) == 0; ch = (s3 - 1) / 2 + (upw ? 1 : 0); }
        if (upw) { int ntl; split(i, ntl, c); src = b.ffn0_w; ld = D; n = 32 * ch + 16 * ntl + n16; }
        else { src = b.ffn2_w; ld = a.F; n = 16 * i + n16; c = 0; kbase = 32 * ch; }
    }
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = src[(int64_t)n * ld + kbase + bperm_k(c, gg, j)];
    uint4 o;
    o.x = bpack2<DT>(v[0], v[1]); o.y = bpack2<DT>(v[2], v[3]); o.z = bpack2<DT>(v[4], v[5]); o.w = bpack2<DT>(v[6], v[7]);
    static_cast<uint4*>(a.frags)[(int64_t)f * 64 + lane] = o;
}

template <int D>
__global__ __launch_bounds__(256) void blocks_pack_vec_kernel(BlkPackArgs a) {
    typedef Geo<D> G;
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int lvs = G::lv_size(a.F);
    if (i >= a.n_layers * lvs) return;
    const int l = i / lvs, r = i % lvs;
    const auto& b = a.p.blk[l];
    float v;
    if (r < G::B1) {
        const float* srcs[8] = {b.ln_attn_w, b.ln_attn_b, b.q_b, b.k_b, b.v_b, b.out_b, b.ln_ffn_w, b.ln_ffn_b};
        v = srcs[r / D][r % D];
    } else if (r < G::b2(a.F)) v = b.ffn0_b[r - G::B1];
    else v = b.ffn2_b[r - G::b2(a.F)];
    a.vec[i] = v;
}

constexpr int LDS_STATIC_MAX = 2 * 16 * 1024 + 2 * 4 * 2 * 3 * 64 * 8;      // upper bound of ring + K/V exchange over the shapes

bool blocks_shape_ok(const bsrl_blocks_desc* d) {
    if (!d) return false;
    const bool geo = (d->d == 128 && d->n_heads == 4) || (d->d == 192 && d->n_heads == 4) || (d->d == 256 && d->n_heads == 8);
    if (!geo || d->T < 1 || d->T > 32 || d->ffn <= 0 || d->ffn % 32 != 0 || d->ffn < 64 || d->n_layers < 1 ||
        d->n_layers > BSRL_MAX_LAYERS || (d->dtype != BSRL_F16 && d->dtype != BSRL_BF16) ||
        (d->act != BSRL_ACT_RELU && d->act != BSRL_ACT_GELU) || d->n_queries < 0 || d->n_queries > 16 || d->n_queries > d->T)
        return false;
    const int64_t vec_bytes = (int64_t)d->n_layers * (9 * d->d + d->ffn) * 4;
    return vec_bytes + LDS_STATIC_MAX <= LDS_BUDGET;
}
int64_t blocks_stages(const bsrl_blocks_desc* d) {
    return (int64_t)d->n_layers * (d->d == 128 ? Geo<128>::layer_stages(d->ffn) : d->d == 192 ? Geo<192>::layer_stages(d->ffn) : Geo<256>::layer_stages(d->ffn));
}
int64_t blocks_frag_bytes(const bsrl_blocks_desc* d) { return blocks_stages(d) * (d->d / 16) * 1024; }

template <typename DT, int D, int DH>
void pack_launch(const BlkPackArgs& pa, int64_t nfrags, hipStream_t st) {
    hipLaunchKernelGGL((blocks_pack_frags_kernel<DT, D, DH>), dim3((unsigned)((nfrags + 3) / 4)), dim3(256), 0, st, pa);
    const int nvec = pa.n_layers * Geo<D>::lv_size(pa.F);
    hipLaunchKernelGGL(blocks_pack_vec_kernel<D>, dim3((unsigned)((nvec + 255) / 256)), dim3(256), 0, st, pa);
}

// dynamic LDS of the env-per-wave kernel: vectors (rounded to 1 KB) + ring
template <int D> size_t env_dyn_bytes(int n_layers, int F) {
    return (size_t)((n_layers * Geo<D>::lv_size(F) / 4 + 63) & ~63) * 16 + (size_t)EnvRing<D>::SLOTS * EnvRing<D>::STAGE_BYTES;
}
// The env-per-wave kernel runs where a wave's state fits 256 registers (d = 128 and 192: at d = 256 it would spill
// several hundred values), the vectors and the stage ring fit a workgroup's LDS, and the stack is at least as long as
// the ring; the wave-pair kernel otherwise.
template <int D> bool env_kernel_ok(const BlkArgs& a) {
    if (D == 256) return false;
    return env_dyn_bytes<D>(a.n_layers, a.F) + 1024 <= (size_t)LDS_BUDGET && a.total_stages >= EnvRing<D>::SLOTS && a.total_stages % 2 == 0;
}

template <typename DT, int D, int DH, int ACT>
int fwd_launch(const BlkArgs& a_, int cus, hipStream_t st) {
    BlkArgs a = a_;
    if constexpr (D != 256) {
        // Few envs: one per workgroup, its features over the waves (blocks_latency.hip).  us at d = 192, six blocks | d = 128, three,
        // with it / without: 1 env 68 / 206 | 18 / 41, 256 envs 76 / 216 | 22 / 44, 512 (two rounds) 148 / 216 | 41 / 47,
        // 1024 321 / 246 | 86 / 54.  All three kernels produce the same bits for an env.
        if (a.B <= 2 * (int64_t)cus) {
            const BlocksLatencyArgs l{reinterpret_cast<const uint4*>(a.frags), a.vec, a.x_in, a.key_bias, a.x_res, a.x_out, a.B, a.n_layers, a.F, a.T, a.n_queries};
            if (bsrl_blocks_latency(l, D, ACT, std::is_same<DT, F16>::value ? BSRL_F16 : BSRL_BF16, cus, st)) return BSRL_OK;
        }
        // d = 192 up to 4 envs per CU: the wave-pair kernel's row tile per wave has the shorter chain (1024 envs 246 against 254 us;
        // at d = 128 it is 65 against 54)
        if (env_kernel_ok<D>(a) && (D == 128 || a.B > 4 * (int64_t)cus)) {
            const size_t dyn = env_dyn_bytes<D>(a.n_layers, a.F);
            // as few envs per workgroup as the rounds over the CUs allow: a wave alone on its SIMD shares it with nobody
            // (1500 envs at d = 192: 327 -> 306 us)
            const int64_t rounds = (a.B + (int64_t)EnvRing<D>::NW * cus - 1) / ((int64_t)EnvRing<D>::NW * cus);
            a.per = (int)((a.B + rounds * cus - 1) / (rounds * cus));
            const int64_t ntiles = (a.B + a.per - 1) / a.per;
            auto kern = blocks_env_kernel<DT, D, DH, ACT>;
            if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) != hipSuccess)
                return BSRL_UNSUPPORTED;
            hipLaunchKernelGGL(kern, dim3((unsigned)(ntiles < cus ? ntiles : cus)), dim3(EnvRing<D>::NW * 64), dyn, st, a);
            return BSRL_OK;
        }
    }
    const size_t dyn = (size_t)a.n_layers * Geo<D>::lv_size(a.F) * sizeof(float);
    const int64_t ntiles = (a.B + 3) / 4;
    const dim3 grid((unsigned)(ntiles < cus ? ntiles : cus));
    auto kern = blocks_kernel<DT, D, DH, ACT>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) != hipSuccess)
        return BSRL_UNSUPPORTED;
    hipLaunchKernelGGL(kern, grid, dim3(512), dyn, st, a);
    return BSRL_OK;
}

}  // namespace

extern "C" int64_t bsrl_blocks_pack_size(const bsrl_blocks_desc* d) {
    if (!blocks_shape_ok(d)) return 0;
    return blocks_frag_bytes(d) + (int64_t)d->n_layers * (9 * d->d + d->ffn) * 4;
}

extern "C" int bsrl_blocks_pack(const bsrl_blocks_desc* d, const bsrl_blocks_params* p, void* packed, bsrl_stream stream) {
    if (!d || !p || !packed) BSRL_FAIL(BSRL_EINVAL, "bsrl_blocks_pack: null pointer");
    if (!blocks_shape_ok(d)) return BSRL_UNSUPPORTED;
    if (!bsrl_aligned(packed, 16)) BSRL_FAIL(BSRL_EINVAL, "bsrl_blocks_pack: image must be 16-byte aligned");
    for (int l = 0; l < d->n_layers; ++l) {
        const float* const* ptrs = reinterpret_cast<const float* const*>(&p->blk[l]);
        for (int i = 0; i < 16; ++i)
            if (!ptrs[i]) BSRL_FAIL(BSRL_EINVAL, "bsrl_blocks_pack: null parameter pointer in block %d", l);
    }
    BlkPackArgs pa;
    pa.p = *p; pa.frags = packed;
    pa.vec = reinterpret_cast<float*>(static_cast<char*>(packed) + blocks_frag_bytes(d));
    pa.n_layers = d->n_layers; pa.F = d->ffn;
    const int64_t nfrags = blocks_stages(d) * (d->d / 16);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (d->d == 128) { if (d->dtype == BSRL_F16) pack_launch<F16, 128, 32>(pa, nfrags, st); else pack_launch<BF16, 128, 32>(pa, nfrags, st); }
    else if (d->d == 256) { if (d->dtype == BSRL_F16) pack_launch<F16, 256, 32>(pa, nfrags, st); else pack_launch<BF16, 256, 32>(pa, nfrags, st); }
    else { if (d->dtype == BSRL_F16) pack_launch<F16, 192, 48>(pa, nfrags, st); else pack_launch<BF16, 192, 48>(pa, nfrags, st); }
    BSRL_CHECK_LAUNCH("bsrl_blocks_pack");
    return BSRL_OK;
}

extern "C" int bsrl_blocks_forward(const bsrl_blocks_desc* d, const void* packed, const void* x_in, const void* key_bias,
                                   void* x_res, void* x_out, int64_t B, bsrl_stream stream) {
    return bsrl_blocks_unless(d, packed, x_in, key_bias, x_res, x_out, B, nullptr, stream);
}

int bsrl_blocks_unless(const bsrl_blocks_desc* d, const void* packed, const void* x_in, const void* key_bias, void* x_res, void* x_out, int64_t B,
                       const BlocksPairPlan* plan, bsrl_stream stream) {
    if (!d || !packed || !x_in || !key_bias || !x_out) BSRL_FAIL(BSRL_EINVAL, "bsrl_blocks_forward: null pointer");
    if (!blocks_shape_ok(d)) return BSRL_UNSUPPORTED;
    if (B < 0) BSRL_FAIL(BSRL_EINVAL, "bsrl_blocks_forward: B < 0");
    if (!bsrl_aligned(packed, 16) || !bsrl_aligned(x_in, 8) || !bsrl_aligned(x_out, 8) || (x_res && !bsrl_aligned(x_res, 8)))
        BSRL_FAIL(BSRL_EINVAL, "bsrl_blocks_forward: image must be 16-byte, token streams 8-byte aligned");
    if (B == 0) return BSRL_OK;
    BlkArgs a;
    a.frags = static_cast<const uint2*>(packed);
    a.vec = reinterpret_cast<const float*>(static_cast<const char*>(packed) + blocks_frag_bytes(d));
    a.x_in = static_cast<const u16*>(x_in); a.key_bias = static_cast<const u16*>(key_bias);
    a.x_res = static_cast<u16*>(x_res); a.x_out = static_cast<u16*>(x_out);
    a.B = B; a.n_layers = d->n_layers; a.F = d->ffn; a.T = d->T; a.n_queries = d->n_queries;
    a.total_stages = (int)blocks_stages(d);
    a.plan = plan ? *plan : BlocksPairPlan{};
    hipStream_t st = static_cast<hipStream_t>(stream);
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    int rc;
    const bool relu = d->act == BSRL_ACT_RELU, f16 = d->dtype == BSRL_F16;
    if (d->d == 128) {
        if (f16) rc = relu ? fwd_launch<F16, 128, 32, BSRL_ACT_RELU>(a, cus, st) : fwd_launch<F16, 128, 32, BSRL_ACT_GELU>(a, cus, st);
        else rc = relu ? fwd_launch<BF16, 128, 32, BSRL_ACT_RELU>(a, cus, st) : fwd_launch<BF16, 128, 32, BSRL_ACT_GELU>(a, cus, st);
    } else if (d->d == 256) {
        if (f16) rc = relu ? fwd_launch<F16, 256, 32, BSRL_ACT_RELU>(a, cus, st) : fwd_launch<F16, 256, 32, BSRL_ACT_GELU>(a, cus, st);
        else rc = relu ? fwd_launch<BF16, 256, 32, BSRL_ACT_RELU>(a, cus, st) : fwd_launch<BF16, 256, 32, BSRL_ACT_GELU>(a, cus, st);
    } else {
        if (f16) rc = relu ? fwd_launch<F16, 192, 48, BSRL_ACT_RELU>(a, cus, st) : fwd_launch<F16, 192, 48, BSRL_ACT_GELU>(a, cus, st);
        else rc = relu ? fwd_launch<BF16, 192, 48, BSRL_ACT_RELU>(a, cus, st) : fwd_launch<BF16, 192, 48, BSRL_ACT_GELU>(a, cus, st);
    }
    if (rc != BSRL_OK) return rc;
    BSRL_CHECK_LAUNCH("bsrl_blocks_forward");
    return BSRL_OK;
}
