// latent_step.h — latent attention of single tokens (latent_step.hip), as latent_attn.hip calls it.
#pragma once
#include "../../include/hydra_mix.h"

namespace hxm {

// For arguments that the wide forms take (sizes, strides, alignment): batches in which a sequence brings one token at most.
bool latent_step_serves(const hxm_latent_attn_args& a);
int latent_step_splits(const hxm_latent_attn_args& a);
int launch_latent_step(const hxm_latent_attn_args& a, hipStream_t s);

}  // namespace hxm
