// The fp32 backward at head size 64.
#include "f32_launch.h"

namespace arhip {

void launch_f32_bwd_64(hipStream_t stream, const FlashBwdParams &p, bool causal, BwdForm form) { launch_bwd<64, false>(stream, p, causal, form); }

}  // namespace arhip
