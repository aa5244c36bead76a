// The fp32 forward with an additive mask, in a translation unit of its own so that it compiles beside the plain one.
#include "flash_f32.h"
#include "f32_launch.h"

namespace arhip {
namespace {
template <int D, int QW, int KW>
void go(hipStream_t stream, const FlashF32Params &p, bool causal)
{
    const dim3 grid((unsigned)p.total), block(QW * KW * 64);
    if (causal) hipLaunchKernelGGL((flash_f32_kernel<D, QW, KW, true, true>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((flash_f32_kernel<D, QW, KW, false, true>), grid, block, 0, stream, p);
}
template <int D>
void forms(hipStream_t stream, const FlashF32Params &p, bool causal, int form)
{
    if (form == 81) go<D, 8, 1>(stream, p, causal);
    else if (form == 41) go<D, 4, 1>(stream, p, causal);
    else go<D, 1, 4>(stream, p, causal);
}
}  // namespace

void launch_f32_mask(hipStream_t stream, const FlashF32Params &p, int D, bool causal, int form)
{
    if (D == 64) forms<64>(stream, p, causal, form);
    else forms<128>(stream, p, causal, form);
}
}  // namespace arhip
