// The pipelined attention kernel on bf16 operands with an additive mask: 4 waves at head size 64 (two workgroups per
// compute unit), 8 or 4 at 128.
#include "attn_pipe.h"
#include "pipe_launch.h"

namespace arhip {
namespace {
template <int D, int NW>
void go(hipStream_t stream, const AttnParams &p, bool causal)
{
    const dim3 grid((unsigned)p.total), block(NW * 64);
    if (causal) hipLaunchKernelGGL((attn_pipe_kernel<D, true, MODE_BF16, false, NW, false, false, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((attn_pipe_kernel<D, false, MODE_BF16, false, NW, false, false, true>), grid, block, 0, stream, p);
}
}  // namespace

void launch_pipe_bf16_mask(hipStream_t stream, const AttnParams &p, int D, bool causal, int nw)
{
    if (D == 64) go<64, 4>(stream, p, causal);
    else if (nw == 4) go<128, 4>(stream, p, causal);
    else go<128, 8>(stream, p, causal);
}
}  // namespace arhip
