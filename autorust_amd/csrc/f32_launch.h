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
// Form 14: whether Q is read by whole rows and turned around (RowTurn), or by the lanes that own its rows.  Turning has a price that does not go
// by the number of rows; lanes that own fewer rows touch fewer lines.  Under the causal mask, where all workgroups run at once, the others wait
// for the last one, so it goes by the rows of that one where it is the only one whose waves take another round of key tiles (the first rows
// of every 128), at head size 128 also where hardly a wave takes two tiles, and where some 30 short ones more than run at once are left for a
// second round.
// Without the causal mask the workgroups are alike: rows of lanes on heads of one key tile and on long ones at head size 128, on those of
// two tiles to a wave, and all longer ones with a mask, at 64.  More workgroups than run at once are turned there throughout: two on a compute
// unit, whose loads the L1 has to serve at a time.
// us, by rows of lanes / turned.  Head size 128: B3 H32 N18 7.9 / 8.6, B1 H24 N36 8.9 / 8.8, H8 N50 masked 9.0 / 9.2, H32 N100 11.4 / 10.7, B2 H12 N197
// 14.7 / 13.9, H4 N1000 30.0 / 30.0, N2048 52 / 54, causal B8 H12 N20 8.2 / 8.9, H8 N41 8.4 / 8.9, N64 9.4 / 9.4, N80 9.5 / 9.7, N96 10.3 / 9.9,
// N257 15.1 / 15.6, N272 16.2 / 16.1, N500 20.6 / 19.2, H4 N2048 58 / 50.  Head size 64: H8 N32 5.9 / 5.6, N150 7.9 / 7.9, N224 7.9 / 8.0,
// N256 7.9 / 8.0, N280 9.3 / 9.4, N600 13.0 / 12.4, H12 N544 masked 15.1 / 15.7, causal H8 N32 6.3 / 5.9, N129 7.5 / 7.8, N150 7.9 / 8.1, N160
// 8.2 / 8.1, N257 9.1 / 9.3, N385 10.4 / 10.8, N528 12.1 / 12.2, N536 12.6 / 12.3, N641 13.3 / 13.5, N800 16.4 / 15.4.  More than 256 workgroups:
// head size 64, H40 N222 (280) 12.0 / 11.0, masked 12.8 / 11.8, causal H20 N400 (260) 11.9 / 11.1, H16 N528 (272) 13.7 / 12.6; head size 128,
// causal, H29 N270 (261) 17.9 / 18.8, H27 N320 (270) 19.5 / 19.0, H28 N320 (280) 17.7 / 18.0, H32 N270 (288) 17.3 / 17.9, H36 N240 (288) 17.7 / 18.3,
// N300 (360) 23.3 / 22.5, H12 N710 (276) 26.5 / 24.6.
inline bool f32_turn(int D, int N, int workgroups, bool causal, bool masked)
{
    const int into_round = (N - 1) % (4 * F32_BK) + 1;
    if (D == 64 && N > 128 && workgroups > 256) return true;
    if (!causal) return D == 64 ? N <= 160 || (N > 288 && !masked) : N > (masked ? 64 : F32_BK) && N < 1000;
    if (N > 128 && workgroups > 272) return workgroups > 300 || N > 320;
    if (D == 64) return N <= 128 || N >= 768 || into_round > (N < 512 ? 24 : 16);
    return N > 84 && (N <= 128 || N >= 512 || into_round > (workgroups > 256 ? 24 : 10));
}

// tile_sums: of form 81 at head size 128 (f32_tile_sums)
template <int D, bool HAS_MASK>
void launch_f32_forms(hipStream_t stream, const FlashF32Params &p, bool causal, int form, bool tile_sums)
{
    if (D == 64 && form == 42) launch_f32_form<D, 4, D == 64 ? 2 : 1, HAS_MASK, false>(stream, p, causal);
    else if (form == 14 && !f32_turn(D, p.N, p.total, causal, HAS_MASK)) launch_f32_form<D, 1, 4, HAS_MASK, false, false>(stream, p, causal);
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
