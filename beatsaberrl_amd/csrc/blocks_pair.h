// The block stack over the attendable tokens of two envs per wave (blocks_pair.hip), launched by note_forward.hip.
#pragma once
#include "bsrl_common.h"

constexpr int BLOCKS_PAIR_CHUNK = 64;                // envs that are paired among each other

// What the device found out about a batch: groups of four waves' work per chunk; and what a round of either kernel takes
struct BlocksPairPlan { int* tiles; int chunks, cus; int64_t B; int pair_ns, env_ns; };

__device__ __forceinline__ int blocks_pair_tiles(const BlocksPairPlan& p, int lane) {
    int n = 0;
    for (int c = lane; c < p.chunks; c += WAVE) n += p.tiles[c];
#pragma unroll
    for (int o = 1; o < WAVE; o *= 2) n += __shfl_xor(n, o, WAVE);
    return __builtin_amdgcn_readfirstlane(n);
}
// A round of the pair kernel (a tile per CU) and one of blocks_env_kernel (8 envs per CU), in ns: the attention of two envs at once
// weighs more than one's, the FFN less, so that it is the FFN's width that decides.  d = 192, f16, 16384 envs (8 rounds of either), whole
// stack, us, pairs / one env per wave: one block F = 192 396 / 423, 384 415 / 469, 768 453 / 550; two blocks 673 / 679, 731 / 787, 847 /
// 1004; six 1719 / 1646, 1926 / 2003, 2339 / 2726.
inline BlocksPairPlan blocks_pair_plan(int* tiles, int chunks, int cus, int64_t B, int n_layers, int F) {
    const int full = n_layers - 1;                   // the final block's queries are the lead tokens
    return {tiles, chunks, cus, B, full * (28000 + 24 * F) + 25800 + 12 * F, full * (22500 + 41 * F) + 26500 + 27 * F};
}
__host__ __device__ inline bool blocks_pairs_pay(const BlocksPairPlan& p, int64_t ntiles) {
    const int64_t pairs = (ntiles + p.cus - 1) / p.cus, envs = (p.B + 8 * p.cus - 1) / (8 * p.cus);
    return p.env_ns == 0 || pairs * p.pair_ns <= envs * p.env_ns;
}

// entry of `pairs`: ids of two envs and their attendable optional tokens (bit t: token lead + t)
struct BlocksPairArgs {
    const uint4* frags; const float* vec;            // bsrl_blocks_pack's image
    const u16* x_in; const u16* key_bias; u16* x_res; u16* x_out;
    int4* pairs;                                     // a chunk's worth of entries per chunk; like plan.tiles written by the launch
    BlocksPairPlan plan;
    int n_layers, F, T, lead, total_stages;
};
inline int64_t bsrl_blocks_pair_chunks(int64_t B) { return (B + BLOCKS_PAIR_CHUNK - 1) / BLOCKS_PAIR_CHUNK; }
// bsrl_blocks_forward with n_queries = lead, ReLU, where every token past the first `lead` whose key bias says that attention
// cannot see it (below -BSRL_MASK_BIAS / 2) may be left out: its rows of x_res are zero, everything else has the same bits.
// To be followed by bsrl_blocks_unless with the same plan, which does the batch where pairs do not pay.
// BSRL_UNSUPPORTED, and nothing launched: outside what it covers (d = 192, lead <= 5, T - lead <= 24, more than 4 envs per CU), or
// where pairs cannot pay
int bsrl_blocks_pair(const BlocksPairArgs& a, int d, int dtype, hipStream_t st);
// bsrl_blocks_forward; with a plan, kernels that return at once where pairs pay
int bsrl_blocks_unless(const bsrl_blocks_desc* d, const void* packed, const void* x_in, const void* key_bias, void* x_res, void* x_out, int64_t B,
                       const BlocksPairPlan* plan, bsrl_stream stream);

// What the update's backward reads of a block (note_train.hip), written by the stack itself: rows of the update's compacted stream, token t
// < lead of env b at lead b + t, its i-th attendable note at lead B + noff[b] + i.  x, h: the block's input and its LayerNorm; qkv: q, k, v
// (k, v in the final block, q by itself: its lead rows), each head after head, a head's rows (d / heads wide) one after another - a whole line
// at a time, where rows of all heads took its 96 bytes each at a time: 4.1 -> 3.65 ms for the recipe's 16384 envs -, v without its bias; att: attention's output; xm, h2, hid: the stream behind it, its
// LayerNorm, the FFN's hidden; mean, rstd: of the two LayerNorms.  In the final block q, att and what follows are the lead rows'.  lead: the
// stack's output rows once more, beside the workspace's, from which the rollout's own readout goes on.
struct BlocksSaveLayer { u16 *x, *h, *qkv, *q, *att, *xm, *h2, *hid; float *mean1, *rstd1, *mean2, *rstd2; };
struct BlocksSave { const int32_t* noff; u16* lead; uint32_t rows; BlocksSaveLayer blk[BSRL_MAX_LAYERS]; };       // rows: what every buffer has room for
// bsrl_blocks_pair that saves them, over every env, whether pairs pay or not
bool bsrl_blocks_pair_saves(int64_t B, int d, int heads, int F, int T, int cus);
int bsrl_blocks_pair_save(const BlocksPairArgs& a, const BlocksSave& save, int dtype, hipStream_t st);
