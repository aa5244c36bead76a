// Launchers of the fp32 forward and backward, each in a translation unit of its own so that they compile side by side (f32_fwd_*.hip,
// f32_mask.hip, f32_bwd_*.hip).  p.total workgroups; form: 81, 41, 14 or, head size 64, 42, the tiling (blocks of 32 queries, groups of key tiles).
#pragma once

#include "flash_bwd_f32.h"

namespace arhip {

template <int D, int QW, int KW, bool HAS_MASK, bool TILE_SUMS, bool TURN = (KW > 1)>
void launch_f32_form(hipStream_t stream, const FlashF32Params &p, bool causal)
{
    const dim3 grid((unsigned)p.total), block(QW * KW * 64);
    if (causal) hipLaunchKernelGGL((flash_f32_kernel<D, QW, KW, true, HAS_MASK, TILE_SUMS, TURN>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((flash_f32_kernel<D, QW, KW, false, HAS_MASK, TILE_SUMS, TURN>), grid, block, 0, stream, p);
}
// Form 14 at head size 128: whether Q is read by whole rows and turned around (at head size 64 it always is).  Heads of one key tile are too short for
// the code it takes, and long ones that are not causal have no use for it.  us, by rows of lanes / turned: B3 H32 N18 7.9 / 8.6, B8 H12 N20 causal 8.2
// / 8.9, B1 H24 N36 8.9 / 8.8, H32 N100 11.4 / 10.7, B2 H12 N197 14.7 / 13.9, H8 N500 causal 20.6 / 19.4, H4 N1000 30.0 / 30.0, causal
// 31.6 / 29.1, H4 N2048 52 / 54, causal 58 / 50.
inline bool f32_turn_128(int N, bool causal) { return N > F32_BK && (causal || N < 1000); }

// tile_sums: of form 81 at head size 128 (f32_tile_sums)
template <int D, bool HAS_MASK>
void launch_f32_forms(hipStream_t stream, const FlashF32Params &p, bool causal, int form, bool tile_sums)
{
    if (D == 64 && form == 42) launch_f32_form<D, 4, D == 64 ? 2 : 1, HAS_MASK, false>(stream, p, causal);
    else if (D == 128 && form == 14 && !f32_turn_128(p.N, causal)) launch_f32_form<D, 1, 4, HAS_MASK, false, D != 128>(stream, p, causal);
    else if (form == 14) launch_f32_form<D, 1, 4, HAS_MASK, false>(stream, p, causal);
    else if (form == 41) launch_f32_form<D, 4, 1, HAS_MASK, false>(stream, p, causal);
    else if (D == 128 && tile_sums) launch_f32_form<D, 8, 1, HAS_MASK, D == 128>(stream, p, causal);
    else launch_f32_form<D, 8, 1, HAS_MASK, false>(stream, p, causal);
}

void launch_f32_64(hipStream_t stream, const FlashF32Params &p, bool causal, int form);
void launch_f32_128(hipStream_t stream, const FlashF32Params &p, bool causal, int form, bool tile_sums);
void launch_f32_mask(hipStream_t stream, const FlashF32Params &p, int D, bool causal, int form, bool tile_sums);
void launch_f32_bwd_64(hipStream_t stream, const FlashBwdParams &p, bool causal, BwdForm form);
void launch_f32_bwd_128(hipStream_t stream, const FlashBwdParams &p, bool causal, BwdForm form);
void launch_f32_bwd_mask(hipStream_t stream, const FlashBwdParams &p, int D, bool causal, BwdForm form);

}  // namespace arhip
