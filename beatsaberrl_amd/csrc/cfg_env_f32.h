// The benchmark-config forward in fp32 with an env's rows in LDS from tokenizer to logits (cfg_env_f32.hip), launched by
// bsrl_cfg_rows_forward.
#pragma once
#include "bsrl_common.h"

struct CfgEnvF32Args {
    bsrl_cfg_rows_weights w;                         // lead_img: the packed weights
    const float* obs; int64_t obs_ld;
    const int32_t* n_valid; float *logits, *value;
    int B, n_layers, T, n_out, final_ln, prop_dim, obj_dim;
};
// The image's bytes, 0 where the kernel does not cover the model; the image of w's matrices; the forward (false: not launched)
int64_t bsrl_cfg_env_f32_pack_size(const bsrl_cfg_desc* d);
int bsrl_cfg_env_f32_pack(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w, void* img, hipStream_t st);
bool bsrl_cfg_env_f32(const bsrl_cfg_desc* d, const CfgEnvF32Args& a, hipStream_t st);
