// The benchmark-config forward of few envs at d = 384 (cfg_env_rows.hip), launched by bsrl_cfg_rows_forward.
#pragma once
#include "bsrl_common.h"

struct CfgEnvRowsArgs {
    bsrl_cfg_rows_weights w;                         // lead_img: the packed weights
    const void* obs; int64_t obs_ld;
    const int32_t* noff;                             // prefix sums of the attendable objects, (B + 1)
    u16* x1; float* part;                            // (B T, d); 4 x (B T, d)
    float *logits, *value;
    int B, n_layers, T, n_out, final_ln, prop_dim, obj_dim, obs_f32;
};
// The image's bytes, 0 where the kernels do not cover the model; the image of w's matrices; whether the forward takes these weights; the forward
int64_t bsrl_cfg_env_rows_pack_size(const bsrl_cfg_desc* d);
int bsrl_cfg_env_rows_pack(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w, void* img, hipStream_t st);
bool bsrl_cfg_env_rows_ok(const bsrl_cfg_desc* d, const bsrl_cfg_rows_weights* w);
int bsrl_cfg_env_rows(const bsrl_cfg_desc* d, const CfgEnvRowsArgs& a, hipStream_t st);
