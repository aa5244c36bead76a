// The fp32 backward with an additive mask, in a translation unit of its own so that it compiles beside the plain one.
#include "f32_launch.h"

namespace arhip {

void launch_f32_bwd_mask(hipStream_t stream, const FlashBwdParams &p, int D, bool causal, bool split)
{
    launch_bwd<true>(stream, p, D, causal, split);
}

}  // namespace arhip
