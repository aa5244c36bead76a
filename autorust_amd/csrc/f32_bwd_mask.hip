// The fp32 backward with an additive mask.
#include "f32_launch.h"

namespace arhip {

void launch_f32_bwd_mask(hipStream_t stream, const FlashBwdParams &p, int D, bool causal, BwdForm form)
{
    if (D == 64) launch_bwd<64, true>(stream, p, causal, form);
    else launch_bwd<128, true>(stream, p, causal, form);
}

}  // namespace arhip
