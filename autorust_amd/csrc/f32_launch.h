// Launchers of the fp32 forward and backward with an additive mask (f32_mask.hip, f32_bwd_mask.hip).  p.total workgroups; form: 81, 41 or 14, the tiling
// (blocks of 32 queries, groups of key tiles).
#pragma once

#include "flash_bwd_f32.h"

namespace arhip {

void launch_f32_mask(hipStream_t stream, const FlashF32Params &p, int D, bool causal, int form, bool tile_sums);
void launch_f32_bwd_mask(hipStream_t stream, const FlashBwdParams &p, int D, bool causal, bool split);

}  // namespace arhip
