// The block stack over the attendable tokens of two envs per wave (blocks_pair.hip), launched by note_forward.hip.
#pragma once
#include "bsrl_common.h"

constexpr int BLOCKS_PAIR_CHUNK = 64;                // envs that are paired among each other

// What the device found out about a batch: groups of four waves' work per chunk
struct BlocksPairPlan { int* tiles; int chunks, cus; int64_t B; };

__device__ __forceinline__ int blocks_pair_tiles(const BlocksPairPlan& p, int lane) {
    int n = 0;
    for (int c = lane; c < p.chunks; c += WAVE) n += p.tiles[c];
#pragma unroll
    for (int o = 1; o < WAVE; o *= 2) n += __shfl_xor(n, o, WAVE);
    return __builtin_amdgcn_readfirstlane(n);
}
// A round of the pair kernel (a tile per CU) takes 245 us at the recipe's shape (d = 192, six blocks, F = 768), one of blocks_env_kernel
// (8 envs per CU) 300.
__device__ __forceinline__ bool blocks_pairs_pay(const BlocksPairPlan& p, int ntiles) {
    const int64_t pairs = (ntiles + p.cus - 1) / p.cus, envs = (p.B + 8 * p.cus - 1) / (8 * p.cus);
    return 5 * pairs <= 6 * envs;
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
// BSRL_UNSUPPORTED, and nothing launched: outside what it covers (d = 192, lead <= 5, T - lead <= 24, more than 4 envs per CU)
int bsrl_blocks_pair(const BlocksPairArgs& a, int d, int dtype, hipStream_t st);
// bsrl_blocks_forward; with a plan, kernels that return at once where pairs pay
int bsrl_blocks_unless(const bsrl_blocks_desc* d, const void* packed, const void* x_in, const void* key_bias, void* x_res, void* x_out, int64_t B,
                       const BlocksPairPlan* plan, bsrl_stream stream);
