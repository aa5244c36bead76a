// The fp32 forward with an additive mask, in a translation unit of its own so that it compiles beside the plain one.
#include "flash_f32.h"
#include "f32_launch.h"

namespace arhip {
namespace {
template <int D, int QW, int KW, bool SUMS>
void go(hipStream_t stream, const FlashF32Params &p, bool causal)
{
    const dim3 grid((unsigned)p.total), block(QW * KW * 64);
    if (causal) hipLaunchKernelGGL((flash_f32_kernel<D, QW, KW, true, true, SUMS>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((flash_f32_kernel<D, QW, KW, false, true, SUMS>), grid, block, 0, stream, p);
}
template <int D>
void forms(hipStream_t stream, const FlashF32Params &p, bool causal, int form, bool sums)
{
    if (form == 14) go<D, 1, 4, false>(stream, p, causal);
    else if (form == 81) sums ? go<D, 8, 1, true>(stream, p, causal) : go<D, 8, 1, false>(stream, p, causal);
    else sums ? go<D, 4, 1, true>(stream, p, causal) : go<D, 4, 1, false>(stream, p, causal);
}
}  // namespace

void launch_f32_mask(hipStream_t stream, const FlashF32Params &p, int D, bool causal, int form, bool tile_sums)
{
    if (D == 64) forms<64>(stream, p, causal, form, tile_sums);
    else forms<128>(stream, p, causal, form, tile_sums);
}
}  // namespace arhip
