// The fp32 backward at head size 128.
#include "f32_launch.h"

namespace arhip {

void launch_f32_bwd_128(hipStream_t stream, const FlashBwdParams &p, bool causal, BwdForm form) { launch_bwd<128, false>(stream, p, causal, form); }

}  // namespace arhip
