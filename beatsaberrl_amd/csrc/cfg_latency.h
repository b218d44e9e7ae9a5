// The config-model forward with a workgroup's features dealt over its waves, one to four envs per workgroup (cfg_latency.hip),
// launched by cfg_forward.hip.
#pragma once
#include "bsrl_common.h"

struct CfgLatencyArgs {
    const uint4* frags; const float* vec;            // bsrl_cfg_pack's image and vectors
    const void* obs; int64_t obs_ld; int obs_f32, tok_vec;
    const int32_t* n_valid; float *logits, *value;
    int B, n_layers, n_logits, final_ln, prop_dim, obj_dim;
};
// F = 512, up to four envs per CU
void bsrl_cfg_latency(const CfgLatencyArgs& a, int act, int dtype, hipStream_t st);
