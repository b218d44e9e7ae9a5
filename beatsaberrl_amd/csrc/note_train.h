// The update's saved activations, as the rollout's block stack writes them (note_forward.hip, note_train.hip).
#pragma once
#include "blocks_pair.h"
#include "note_pack.h"

// the update of B envs may take its block stack from the rollout forward (bsrl_note_train_begin / _end)
bool note_train_saves(const bsrl_note_desc& d, int64_t B);
// where the stack puts what the backward reads, in `saved`
BlocksSave note_train_blocks(const bsrl_note_desc& d, int64_t B, void* saved);
