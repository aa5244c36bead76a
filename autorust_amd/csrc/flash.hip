// arhip_flash_fwd / arhip_sage_fwd: argument checks, kernel selection, launch.
//
// Mirrors the reference's launch wrappers: cuda_flash::run_ex
// (src/runtime/cuda_flash.rs:203-254), cuda_flash_bf16::run_ex
// (src/runtime/cuda_flash_bf16.rs:495-548) and cuda_flash_sage::run_ex
// (src/runtime/cuda_flash_sage.rs:452-485).
#include "arhip_internal.h"
#include "attn_fwd.h"
#include "pipe_launch.h"
#include "flash_bwd_f32.h"
#include "f32_launch.h"

#include <algorithm>
#include <cmath>


using namespace arhip;

extern "C" int arhip_attn_supported(int kind, int64_t n, int64_t d, int dtype)
{
    if (n <= 0 || n > (int64_t)1 << 24) return 0;
    if (d != 64 && d != 128) return 0;
    switch (kind) {
    case ARHIP_ATTN_FLASH: return dtype == ARHIP_F32 || dtype == ARHIP_BF16;
    case ARHIP_ATTN_SAGE: return dtype == ARHIP_F32 || dtype == ARHIP_BF16;
    default: return 0;  // SDPA is the caller's general path
    }
}

static int check_common(const char *fn, arhip_device *dev, const void *q, const void *k, const void *v, const void *o,
                        const float *mask, int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D)
{
    ARHIP_REQUIRE(dev != nullptr, "%s: null device", fn);
    ARHIP_REQUIRE(q && k && v && o, "%s: null tensor pointer", fn);
    ARHIP_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && N > 0, "%s: empty shape B=%lld Hq=%lld Hkv=%lld N=%lld", fn,
                  (long long)B, (long long)Hq, (long long)Hkv, (long long)N);
    ARHIP_REQUIRE(Hq % Hkv == 0, "%s: Hq=%lld is not a multiple of Hkv=%lld", fn, (long long)Hq, (long long)Hkv);
    if (D != 64 && D != 128) return arhip_fail(ARHIP_EUNSUPPORTED, "%s: head_dim %lld (64 or 128)", fn, (long long)D);
    // workgroup ids, tile counts and row indices are 32-bit in the kernels
    if (N > ((int64_t)1 << 24) || B * Hq > ((int64_t)1 << 24) || B * Hq * ((N + 31) / 32) > ((int64_t)1 << 30))
        return arhip_fail(ARHIP_EUNSUPPORTED, "%s: shape too large for 32-bit tile indices", fn);
    ARHIP_REQUIRE(arhip_aligned16(q) && arhip_aligned16(k) && arhip_aligned16(v) && arhip_aligned16(o),
                  "%s: q/k/v/o must be 16-byte aligned", fn);
    ARHIP_REQUIRE(mask == nullptr || (reinterpret_cast<uintptr_t>(mask) & 3u) == 0, "%s: mask must be 4-byte aligned", fn);
    return ARHIP_OK;
}

// CAUSAL / HAS_MASK dispatch of the general kernel.
template <int D, int MODE, bool PER_KEY, bool OUT_F32, bool DBG, bool MASKS>
static void launch_attn(hipStream_t stream, const AttnParams &p, bool causal, bool has_mask)
{
    const dim3 grid((unsigned)p.total), block(256);
    if constexpr (MASKS) {
        if (has_mask) {
            if (causal)
                hipLaunchKernelGGL((attn_fwd_kernel<D, true, true, MODE, PER_KEY, OUT_F32, DBG>), grid, block, 0, stream, p);
            else
                hipLaunchKernelGGL((attn_fwd_kernel<D, false, true, MODE, PER_KEY, OUT_F32, DBG>), grid, block, 0, stream, p);
            return;
        }
    }
    if (causal)
        hipLaunchKernelGGL((attn_fwd_kernel<D, true, false, MODE, PER_KEY, OUT_F32, DBG>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((attn_fwd_kernel<D, false, false, MODE, PER_KEY, OUT_F32, DBG>), grid, block, 0, stream, p);
}

// The software-pipelined kernel (no additive mask): 8 waves per workgroup, or 4 (two workgroups per compute
// unit) where a workgroup sees few tiles.  Its variants are compiled in translation units of their own
// (pipe_launch.h).
// Which of the two: 128 queries per workgroup hide a workgroup's prologue and epilogue under its
// neighbour's tiles and fill the chip with fewer heads, but request every K/V tile twice as often and
// keep only one tile in flight.  Two workgroups of equal length that start together stay in step and
// hide nothing, so the gain is in few or unequal workgroups.  Measured at D = 128, bf16 (B4 H32 unless
// noted; 4 waves against 8): causal N = 512 / 1024 / 2048 -15 / -7 / -5 %, B1 H16 N = 2048 causal -25 %,
// B2 H16 N = 1024 -22 %, N = 1024 -4 %; N = 2048 equal; N = 2048 causal with key lengths in [N/2, N]
// (many equal workgroups) +3 %; N = 8192 +3 %, causal N = 32768 +4.5 %.
// At D = 64 (B4 H32): N = 2048 -8 %, N = 8192 -2 %, causal N = 2048 -16 %, causal N = 8192 -4 %: always 4 waves.
// (D = 64 runs three workgroups per compute unit, 168 registers and 40 KB of LDS each: no faster than two on long
// sequences, B16 H24 N140 10.2 -> 9.6 us.)
static bool pipe_wants_4_waves(arhip_device *dev, int64_t heads, int64_t N, int64_t D, bool causal, bool has_len)
{
    if (dev->attn_waves == 8 || dev->attn_waves == 40) return dev->attn_waves == 40;
    if (D == 64) return true;
    if (heads * ((N + 255) / 256) < 2 * (int64_t)dev->cus) return true;
    return N <= 1024 || (N <= 2048 && causal && !has_len);
}

// The pipelined kernel addresses K and V through 32-bit buffer offsets (rows of one head, plus the
// tiles it requests past the end).
static bool pipe_addressable(int64_t N, int64_t kv_token_stride, int64_t elem_bytes)
{
    return (N + 5 * 64) * kv_token_stride * elem_bytes < ((int64_t)1 << 31);
}

// The form of the pipelined kernel (pipe_launch.h).  groups: two groups of waves have one (bf16 without a mask, 8-bit operands with
// scales over whole tiles).
// A grid whose workgroups of 4 waves all run at once leaves a SIMD one wave, or none, for all tiles of a head.  Groups deal the
// tiles out: 64 queries to a workgroup of 2 + 2 waves, half the tiles to each wave, where those all run at once too (bf16 at head
// size 64 two on a compute unit, which pays where the causal mask leaves half of the tiles anyway), else 128 to one of 4 + 4, which
// share a SIMD two by two.  What it costs is joining the sums and more transfers under way, 0.5 to 2 us, so short heads keep the 4 waves.
// us, 4 waves / 4 + 4 / 2 + 2: bf16 head size 64 B4 H12 N250 6.5 / 7.3 / 6.1, B8 H12 N197 6.5 / 7.4 / 7.8, B1 H8 N1024 13.8 / 12.6 / 9.7,
// causal 14.4 / 12.7 / 9.9, B2 H16 N700 11.7 / 11.7 / 12.4, causal 10.8 / 10.3 / 8.9, B1 H16 N2048 24.5 / 22.0 / 24.1, causal 24.9 / 20.5 /
// 16.8, B1 H4 N8192 causal 85.6 / 65.0 / 54.5; 128 B2 H8 N300 9.5 / 10.8 / 9.8, B1 H8 N512 11.5 / 12.6 / 11.2, N1024 18.3 / 18.2 / 16.7, B1 H8
// N2048 31.7 / 29.3 / 27.3, B2 H16 N1000 21.0 / 21.4 / 32.7, B1 H16 N2048 35.9 / 35.5 / 52.5, causal 32.6 / 30.1 / 34.0; int8 head size 64 B2 H12
// N400 9.5 / 10.7 / 9.9, B1 H8 N1024 14.6 / 14.7 / 12.9, B2 H16 N850 13.7 / 14.2 / 23.6, B1 H16 N2048 23.9 / 22.7 / 35.8.
static int pipe_form(arhip_device *dev, int64_t heads, int64_t N, int64_t D, bool bf16, bool causal, bool has_len, bool groups,
                     int64_t kv_token_stride)
{
    if (groups && pipe_addressable(2 * N, kv_token_stride, 2)) {
        if (dev->attn_waves == PIPE_4X2 || dev->attn_waves == PIPE_2X2) return dev->attn_waves;
        const int64_t wgs128 = heads * ((N + 127) / 128), wgs64 = heads * ((N + 63) / 64);
        const bool two = bf16 && D == 64;  // of 2 + 2 waves on a compute unit
        if (dev->attn_waves != 0) {
        } else if (wgs64 <= dev->cus) {
            if (N > (two ? 128 : 511)) return PIPE_2X2;
        } else if (wgs64 <= 2 * (int64_t)dev->cus) {
            if (two && (causal ? N >= 400 : N >= 1024 && wgs128 > dev->cus)) return PIPE_2X2;
            if (wgs128 <= dev->cus && N >= (two ? 700 : 1500)) return PIPE_4X2;
        }
    }
    return pipe_wants_4_waves(dev, heads, N, D, causal, has_len) ? 4 : 8;
}
// queries per workgroup
static int pipe_rows(int form) { return form == 8 ? 256 : form == PIPE_2X2 ? 64 : 128; }

// The same for launches with an additive mask, whose blocks need LDS of their own: at D = 128 one workgroup per compute
// unit in either form, so 8 waves as soon as 4 would not all run at once.
static bool mask_wants_4_waves(arhip_device *dev, int64_t heads, int64_t N, int64_t D)
{
    if (dev->attn_waves == 8 || dev->attn_waves == 40) return D == 64 || dev->attn_waves == 40;
    return D == 64 || heads * ((N + 127) / 128) <= dev->cus;
}

// Which kernel.  The software-pipelined kernel (with 8 or 4 waves per workgroup, pipe_wants_4_waves' choice) wherever it has a
// form: with its 4-wave form it is the fastest kernel down to the shortest sequences (bf16, against the kernels that used to
// serve them: B8 H12 N197 D64 7.8 -> 7.0 us, B4 H16 N256 D128 11.8 -> 9.0 us, B32 H12 N64 D64 9.1 -> 5.6 us, B8 H12 N400 D64
// 27.8 -> 12.9 us).  special: 8-bit launches with an additive mask, K scales over a number of keys that is no power of two or
// the logits export take the general kernel with 4 waves of 32 queries, as do K/V too large for 32-bit offsets.
// (ARHIP_ATTN_WAVES, read once when the device is opened, is a tuning aid.  4: the general
// kernel; 8, 40: the pipelined kernel with 8 / 4 waves, the same bits; 42, 22: with two groups of 4 / 2 waves, whose sums have exponent references of
// their own: bf16 and 8-bit results differ by the rounding of P to bf16, 2^-8 of the largest |V| at most, and so they do with the size of the grid, by
// which pipe_form chooses.)
static bool use_pipe(arhip_device *dev, bool special, int64_t N, int64_t kv_token_stride)
{
    return !special && dev->attn_waves != 4 && pipe_addressable(N, kv_token_stride, 2);
}

// Tiling of the fp32 forward: 8 or 4 waves of 32 queries that share their key tiles (81, 41: 256 and 128 queries per workgroup),
// or 4 waves on the same 32 queries with the key tiles dealt out between them (14), or, head size 64, two groups of 4 waves that share
// every other key tile (42: 128 queries per workgroup).  The one whose busiest compute unit is done
// first, in units of what a workgroup of 8 waves takes for all its tiles.  Head size 64: a pair of 41 on a compute unit takes 1.1, one alone
// 0.7 (one wave per SIMD hides less), a pair of 14 0.57 and one alone 0.3, and one of 42, which joins its sums at the end, 0.53 and what
// that takes of a short head.  Head size 128, where all three have a compute unit to
// themselves: 0.68 and 0.36.  A causal grid runs longest workgroup first: the longest one, or its even share (half of all tiles and
// half a workgroup's) where there are enough to balance, and what that leaves unbalanced.  Up to 128 queries only the waves of a single
// workgroup have any, and 14 is faster as long as all its workgroups run at once.
// us, 81 / 41 / 14, on grids of H heads: head size 64, N2048 H24 91 / 100 / 142, H48 175 / 169 / 272, H8 74 / 63 / 51, N512 H96 28 / 31 / 47,
// H160 54 / 48 / 76, H24 24 / 20 / 18, N200 H160 16 / 18 / 25, H48 15 / 12 / 12, N64 H160 7.2 / 7.0 / 8.7, causal N2048 H48 93 / 100 / 155, H24
// 81 / 70 / 81, N4096 H8 146 / 118 / 100, N200 H96 16 / 13 / 17; head size 128, N2048 H48 297 / 323 / 634, H8 135 / 93 / 106, N512 H160 91 / 98 /
// 200, H24 43 / 31 / 40, N300 H160 64 / 47 / 115, N128 H160 16 / 16 / 35, causal N2048 H32 133 / 126 / 260, N800
// H96 79 / 91 / 178, H24 58 / 44 / 51, N2048 H8 133 / 97 / 65.
// 42 / the best of the others: N800 H24 25 / 28, N1500 H16 40 / 48, N2048 H8 48 / 52, H16 60 / 65, N4096 H8 113 / 123, N200 H128 14.4 / 13.0,
// causal N512 H64 20 / 22, N800 H36 25 / 29, N2048 H16 50 / 57, H32 69 / 77, N4096 H10 98 / 125, H16 123 / 145, N1024 H64 45 / 43, N3000 H24
// 114 / 112, N800 H64 36 / 32: with a mask of half the tiles not beyond what runs at once, or twice that of long heads.
static int f32_form(int64_t heads, int64_t N, int64_t D, bool causal, int cus)
{
    auto tiles = [&](int rows) { return (N + rows - 1) / rows; };
    if (N <= 128) return heads * tiles(32) <= cus ? 14 : D == 64 ? 41 : 81;
    double c81, c41, c14, c42 = 1e9;
    if (causal) {
        auto share = [&](int rows) { return (double)(heads * (tiles(rows) + 1)) / (2 * cus); };
        c81 = std::max(1.0, 1.15 * share(256) + 0.1);
        c41 = std::max(0.7, D == 64 ? 0.57 * share(128) + 0.2 : 0.9 * share(128) + 60.0 / N);
        c14 = D == 64 ? 0.285 * share(32) + std::max(0.08, 60.0 / N) : 0.5 * share(32) + 90.0 / N;
        if (D == 64 && heads * tiles(128) <= (N >= 2048 ? 2 : 1) * (int64_t)cus) c42 = std::max(0.45, 0.4 * share(128) + 0.15) + 50.0 / N;
    } else {
        auto rounds = [&](int rows) { return (int64_t)((heads * tiles(rows) + cus - 1) / cus); };
        auto pairs = [](int64_t n, double pair, double alone) { return pair * (double)(n / 2) + alone * (double)(n % 2); };
        c81 = (double)rounds(256);
        c41 = D == 64 ? pairs(rounds(128), 1.1, 0.7) : 0.68 * (double)rounds(128);
        c14 = D == 64 ? pairs(rounds(32), 0.57, 0.3) : 0.36 * (double)rounds(32);
        if (D == 64) c42 = (0.53 + 70.0 / N) * (double)rounds(128);
    }
    if (c42 < c81 && c42 < c41 && c42 < c14) return 42;
    if (c14 < c41 && c14 < c81) return 14;
    return c81 < c41 ? 81 : 41;
}

// Whether O is rounded once per key tile (TILE_SUMS) rather than with every matrix instruction: form 81 at head size 128, which has
// no registers for more accumulators.  Relative error (2-norm, against float64) at N = 2048, with / without: 3.1e-7 / 5.5e-7.  Grids
// of fewer than two workgroups of 128 queries per compute unit, which may be long heads with nothing else to fill the chip, take it.
static bool f32_tile_sums(int64_t heads, int64_t N, int cus) { return heads * ((N + 127) / 128) < 2 * (int64_t)cus; }

// The fp32 forward in a form; fp: all but the grid
static void launch_f32(arhip_device *dev, FlashF32Params &fp, int64_t heads, int64_t D, bool causal, int form)
{
    const int bq = form / 10 * 32;
    fp.nq = (fp.N + bq - 1) / bq;
    fp.total = (int)(fp.nq * heads);
    fp.lpt_heads = causal ? (int)heads : 0;  // longest query tile first over all heads
    const bool sums = f32_tile_sums(heads, fp.N, dev->cus);
    if (fp.mask != nullptr) launch_f32_mask(dev->stream, fp, (int)D, causal, form, sums);
    else if (D == 64) launch_f32_64(dev->stream, fp, causal, form);
    else launch_f32_128(dev->stream, fp, causal, form, sums);
}

static void dense_strides(long s[3], int64_t H, int64_t N, int64_t D)
{
    s[0] = (long)(H * N * D);
    s[1] = (long)(N * D);
    s[2] = (long)D;
}

extern "C" int arhip_flash_fwd(arhip_device *dev, const void *q, const void *k, const void *v, void *o,
                               const float *mask, const int32_t *kv_len,
                               int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                               int causal, int dtype, float scale, int wait, double *secs)
{
    long qs[3], ks[3];
    dense_strides(qs, Hq, N, D);
    dense_strides(ks, Hkv, N, D);
    const int64_t q64[3] = {qs[0], qs[1], qs[2]}, k64[3] = {ks[0], ks[1], ks[2]};
    return arhip_flash_fwd_strided(dev, q, k, v, o, q64, k64, q64, mask, kv_len, B, Hq, Hkv, N, D, causal, dtype, scale,
                                   wait, secs);
}

extern "C" int arhip_flash_fwd_strided(arhip_device *dev, const void *q, const void *k, const void *v, void *o,
                                       const int64_t q_strides[3], const int64_t kv_strides[3], const int64_t o_strides[3],
                                       const float *mask, const int32_t *kv_len,
                                       int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                                       int causal, int dtype, float scale, int wait, double *secs)
{
    return arhip_flash_fwd_lse(dev, q, k, v, o, nullptr, q_strides, kv_strides, o_strides, mask, kv_len, B, Hq, Hkv, N, D,
                               causal, dtype, scale, wait, secs);
}

extern "C" int arhip_flash_fwd_lse(arhip_device *dev, const void *q, const void *k, const void *v, void *o, float *lse,
                                   const int64_t q_strides[3], const int64_t kv_strides[3], const int64_t o_strides[3],
                                   const float *mask, const int32_t *kv_len,
                                   int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                                   int causal, int dtype, float scale, int wait, double *secs)
{
    if (int rc = check_common("arhip_flash_fwd", dev, q, k, v, o, mask, B, Hq, Hkv, N, D)) return rc;
    ARHIP_REQUIRE(lse == nullptr || (reinterpret_cast<uintptr_t>(lse) & 3u) == 0, "arhip_flash_fwd_lse: lse must be 4-byte aligned");
    ARHIP_REQUIRE(dtype == ARHIP_F32 || dtype == ARHIP_BF16, "arhip_flash_fwd: dtype %d", dtype);
    ARHIP_REQUIRE(q_strides && kv_strides && o_strides, "arhip_flash_fwd_strided: null strides");
    {
        // rows must stay 16-byte aligned and must not overlap: every stride a multiple of 8 elements,
        // the token stride at least D
        const int64_t *all[3] = {q_strides, kv_strides, o_strides};
        for (int t = 0; t < 3; ++t)
            for (int i = 0; i < 3; ++i)
                ARHIP_REQUIRE(all[t][i] >= 0 && all[t][i] % 8 == 0 && (i != 2 || all[t][i] >= D) && (t != 2 || all[t][i] > 0),
                              "arhip_flash_fwd_strided: stride %lld (multiples of 8 elements, token stride >= D, output "
                              "strides > 0 so that output rows cannot alias)",
                              (long long)all[t][i]);
    }
    ARHIP_HIP(hipSetDevice(dev->ordinal));
    arhip_call_timer t{dev, wait, secs};
    t.kernel = (dtype == ARHIP_F32) ? ARHIP_K_FLASH_F32 : ARHIP_K_FLASH_BF16;

    if (dtype == ARHIP_F32) {
        FlashF32Params fp;
        fp.q = (const float *)q; fp.k = (const float *)k; fp.v = (const float *)v; fp.o = (float *)o;
        fp.mask = mask; fp.kv_len = kv_len; fp.lse = lse;
        fp.Hq = (int)Hq; fp.Hkv = (int)Hkv; fp.N = (int)N;
        for (int i = 0; i < 3; ++i) {
            fp.qs[i] = (long)q_strides[i];
            fp.ks[i] = (long)kv_strides[i];
            fp.os[i] = (long)o_strides[i];
        }
        fp.scale = scale;
        if (int rc = t.begin()) return rc;
        launch_f32(dev, fp, B * Hq, D, causal != 0, f32_form(B * Hq, N, D, causal != 0, dev->cus));
        arhip_note_selected(ARHIP_K_FLASH_F32);
        return t.end();
    }

    AttnParams p = {};
    p.q = q; p.k = k; p.v = (const uint16_t *)v; p.o = o;
    p.mask = mask; p.kv_len = kv_len; p.lse = lse;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.N = (int)N;
    for (int i = 0; i < 3; ++i) {
        p.qs[i] = (long)q_strides[i];
        p.ks[i] = (long)kv_strides[i];
        p.vs[i] = (long)kv_strides[i];
        p.os[i] = (long)o_strides[i];
    }
    p.bq = p.bk = 1;
    p.scale = scale;
    const bool c = causal != 0, hm = mask != nullptr;
    const bool pipe = use_pipe(dev, false, N, kv_strides[2]);
    const int nw = !pipe ? 4 : hm ? (mask_wants_4_waves(dev, B * Hq, N, D) ? 4 : 8) : pipe_form(dev, B * Hq, N, D, true, c, kv_len != nullptr, true, kv_strides[2]);
    p.nq = (int)((N + pipe_rows(nw) - 1) / pipe_rows(nw));
    p.total = (int)(p.nq * B * Hq);
    p.lpt = p.total <= 16 * dev->cus;  // few workgroups per CU: balance them globally
    if (int rc = t.begin()) return rc;
    if (pipe) {
        if (hm) launch_pipe_bf16_mask(dev->stream, p, (int)D, c, nw);
        else launch_pipe_bf16(dev->stream, p, (int)D, c, nw);
    } else if (D == 64) {
        launch_attn<64, MODE_BF16, false, false, false, true>(dev->stream, p, c, hm);
    } else {
        launch_attn<128, MODE_BF16, false, false, false, true>(dev->stream, p, c, hm);
    }
    arhip_note_selected(ARHIP_K_FLASH_BF16);
    return t.end();
}

// A pass through the tensor interface with its wait, us, the entry's own kernel / the form chosen here: fp32 head size 64 B8 H6 N789 71 / 50,
// B16 H16 N300 59 / 48, B2 H16 N2048 143 / 113, 128 B1 H8 N1024 65 / 45, B8 H16 N512 causal 66 / 59; bf16 64 B1 H8 N1024 27.7 / 23.4, B1
// H8 N2000 causal 37.8 / 29.2; int8 64 B1 H8 N2000 causal 47.7 / 44.0.
bool arhip_named_form(arhip_device *dev, arhip_named_family family, int rows, bool has_len, const unsigned grid[3], void *const *bufs,
                      const int64_t *vals)
{
    const int64_t heads = grid[1], N = vals[0], D = vals[1], Hq = vals[4], Hkv = vals[5];
    const bool causal = vals[2] != 0, has_mask = vals[3] != 0;
    void *const *rest = bufs + (has_len ? 6 : 5);  // behind Q, K, V, O, M and the lengths
    for (int i = 0; i < 4; ++i)
        if (!arhip_aligned16(bufs[i])) return false;
    if (heads * ((N + 31) / 32) > ((int64_t)1 << 30)) return false;
    const int32_t *kv_len = has_len ? (const int32_t *)bufs[5] : nullptr;
    const float scale = 1.0f / sqrtf((float)D);
    if (family == ARHIP_NAMED_F32 || family == ARHIP_NAMED_F32_LSE) {
        const bool lse = family == ARHIP_NAMED_F32_LSE;  // behind O
        const int form = f32_form(heads, N, D, causal, dev->cus), own = rows == 32 ? 14 : 41;
        // (the entry of both head sizes has registers and LDS for one workgroup on a compute unit, the form of head size 64 for two)
        if (form == own && !(own == 41 && D == 64 && heads * ((N + 127) / 128) > dev->cus)) return false;
        FlashF32Params p = {};
        p.q = (const float *)bufs[0]; p.k = (const float *)bufs[1]; p.v = (const float *)bufs[2]; p.o = (float *)bufs[3];
        p.lse = lse ? (float *)bufs[4] : nullptr;
        p.mask = has_mask ? (const float *)bufs[lse ? 5 : 4] : nullptr;
        p.kv_len = kv_len;
        p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.N = (int)N;
        dense_strides(p.qs, Hq, N, D);
        dense_strides(p.ks, Hkv, N, D);
        dense_strides(p.os, Hq, N, D);
        p.scale = scale;
        launch_f32(dev, p, heads, D, causal, form);
        return true;
    }
    const bool bf16 = family == ARHIP_NAMED_BF16, fused = family == ARHIP_NAMED_I8_QF || family == ARHIP_NAMED_FP8_QF;
    if (!bf16 && vals[7] < 64) return false;  // scales per key
    const int form = pipe_form(dev, heads, N, D, bf16, causal, has_len, true, D);
    if (form != PIPE_4X2 && form != PIPE_2X2) return false;
    AttnParams p = {};
    p.q = bufs[0]; p.k = bufs[1]; p.v = (const uint16_t *)bufs[2]; p.o = bufs[3];
    p.kv_len = kv_len;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.N = (int)N;
    dense_strides(p.qs, Hq, N, D);
    dense_strides(p.ks, Hkv, N, D);
    dense_strides(p.vs, Hkv, N, D);
    dense_strides(p.os, Hq, N, D);
    p.bq = p.bk = 1;
    p.scale = scale;
    if (!bf16) {
        p.bq = (int)vals[6]; p.bk = (int)vals[7];
        while (((int64_t)64 << p.bk_tile_shift) < vals[7]) ++p.bk_tile_shift;
        p.bk_key_shift = -1;
        p.out_f32 = vals[8] != 0;
        if (fused) p.sq_out = (float *)rest[0];
        else p.sq = (const float *)rest[0];
        p.sk = (const float *)rest[1];
    }
    p.nq = (int)((N + pipe_rows(form) - 1) / pipe_rows(form));
    p.total = (int)(p.nq * heads);
    p.lpt = p.total <= 16 * dev->cus;
    if (bf16) launch_pipe_bf16(dev->stream, p, (int)D, causal, form);
    else if (family == ARHIP_NAMED_I8) launch_pipe_i8(dev->stream, p, (int)D, causal, form);
    else if (family == ARHIP_NAMED_FP8) launch_pipe_fp8(dev->stream, p, (int)D, causal, form);
    else if (family == ARHIP_NAMED_I8_QF) launch_pipe_i8_qf(dev->stream, p, (int)D, causal, form);
    else launch_pipe_fp8_qf(dev->stream, p, (int)D, causal, form);
    return true;
}

extern "C" int arhip_sage_fwd(arhip_device *dev, const int8_t *q8, const int8_t *k8,
                              const float *sq, const float *sk, const uint16_t *v, void *o,
                              const float *mask, const int32_t *kv_len,
                              int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                              int64_t bq, int64_t bk, int causal, int out_dtype, float scale,
                              int32_t *dbg_logits, const int32_t dbg_sel[3],
                              int wait, double *secs)
{
    return arhip_sage_fwd_strided(dev, q8, k8, sq, sk, v, o, nullptr, nullptr, mask, kv_len, B, Hq, Hkv, N, D, bq, bk, causal,
                                  out_dtype, scale, dbg_logits, dbg_sel, wait, secs);
}

static int sage_fwd_impl(arhip_device *dev, const int8_t *q8, const int8_t *k8,
                         const float *sq, const float *sk, const uint16_t *v, void *o,
                         const int64_t v_strides[3], const int64_t o_strides[3],
                         const float *mask, const int32_t *kv_len,
                         int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                         int64_t bq, int64_t bk, int causal, int out_dtype, float scale,
                         int32_t *dbg_logits, const int32_t dbg_sel[3], int wait, double *secs, bool fp8)
{
    if (int rc = check_common("arhip_sage_fwd", dev, q8, k8, v, o, mask, B, Hq, Hkv, N, D)) return rc;
    ARHIP_REQUIRE(sq && sk, "arhip_sage_fwd: null scale pointer");
    ARHIP_REQUIRE(bq >= 1 && bk >= 1, "arhip_sage_fwd: block sizes bq=%lld bk=%lld", (long long)bq, (long long)bk);
    ARHIP_REQUIRE(out_dtype == ARHIP_F32 || out_dtype == ARHIP_BF16, "arhip_sage_fwd: out_dtype %d", out_dtype);
    ARHIP_REQUIRE(dbg_logits == nullptr || dbg_sel != nullptr, "arhip_sage_fwd: dbg_logits without dbg_sel");
    ARHIP_REQUIRE(dbg_logits == nullptr || mask == nullptr, "arhip_sage_fwd: the logits export does not take a mask");
    for (int t = 0; t < 2; ++t) {
        const int64_t *st = t == 0 ? v_strides : o_strides;
        if (!st) continue;
        for (int i = 0; i < 3; ++i)
            ARHIP_REQUIRE(st[i] >= 0 && st[i] % 8 == 0 && (i != 2 || st[i] >= D) && (t == 0 || st[i] > 0),
                          "arhip_sage_fwd_strided: stride %lld (multiples of 8 elements, token stride >= D, output strides > 0)",
                          (long long)st[i]);
    }
    ARHIP_HIP(hipSetDevice(dev->ordinal));

    AttnParams p = {};
    p.q = q8; p.k = k8; p.v = v; p.o = o;
    p.mask = mask; p.kv_len = kv_len;
    p.sq = sq; p.sk = sk;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.N = (int)N;
    dense_strides(p.qs, Hq, N, D);
    dense_strides(p.ks, Hkv, N, D);
    dense_strides(p.vs, Hkv, N, D);
    dense_strides(p.os, Hq, N, D);
    for (int i = 0; i < 3; ++i) {
        if (v_strides) p.vs[i] = (long)v_strides[i];
        if (o_strides) p.os[i] = (long)o_strides[i];
    }
    p.bq = (int)bq; p.bk = (int)bk;
    p.scale = scale;
    const bool dbg = dbg_logits != nullptr;
    ARHIP_REQUIRE(!(fp8 && dbg), "arhip_sage_fwd_fp8: the logits export is an int8 facility");
    const bool c = causal != 0, hm = mask != nullptr, f32o = out_dtype == ARHIP_F32;
    p.out_f32 = f32o;
    // K scales that are uniform over a 64-key tile (bk = 64 * 2^n) take the fast kernel; anything
    // else, including the reference's per-key scales (bk == 1), stages the tile's scales in LDS
    int shift = 0;
    while (((int64_t)64 << shift) < bk) ++shift;
    const bool per_key = ((int64_t)64 << shift) != bk;
    p.bk_tile_shift = shift;
    // ... in the general kernel; scales over a power of two of keys below 64 (the reference's bk = 1 among them)
    // have a form of the pipelined kernel that applies them per logit
    int key_shift = 0;
    while (((int64_t)1 << key_shift) < bk) ++key_shift;
    const bool pipe_keys = per_key && ((int64_t)1 << key_shift) == bk;
    p.bk_key_shift = pipe_keys ? key_shift : -1;
    const int64_t kv_token = std::max<int64_t>(D, v_strides ? v_strides[2] : D);
    const bool pipe = use_pipe(dev, hm || (per_key && !pipe_keys) || dbg, N, kv_token);
    const int nw = pipe ? pipe_form(dev, B * Hq, N, D, false, c, kv_len != nullptr, !pipe_keys, kv_token) : 4;
    p.nq = (int)((N + pipe_rows(nw) - 1) / pipe_rows(nw));
    p.total = (int)(p.nq * B * Hq);
    p.lpt = p.total <= 16 * dev->cus;
    if (dbg) {
        p.dbg = dbg_logits;
        p.dbg_bh = dbg_sel[0]; p.dbg_qt = dbg_sel[1]; p.dbg_kt = dbg_sel[2];
        ARHIP_REQUIRE(p.dbg_bh >= 0 && p.dbg_bh < B * Hq && p.dbg_qt >= 0 && (int64_t)p.dbg_qt * 32 < N &&
                          p.dbg_kt >= 0 && (int64_t)p.dbg_kt * 64 < N,
                      "arhip_sage_fwd: debug tile selector out of range");
    }
    arhip_call_timer t{dev, wait, secs};
    t.kernel = ARHIP_K_SAGE;
    if (int rc = t.begin()) return rc;
#define SAGE_V(DD, PK, DB_, MK)                                                                   \
    do {                                                                                               \
        if (f32o) launch_attn<DD, MODE_I8, PK, true, DB_, MK>(dev->stream, p, c, hm);             \
        else launch_attn<DD, MODE_I8, PK, false, DB_, MK>(dev->stream, p, c, hm);                 \
    } while (0)
#define SAGE_D(DD)                                                                                     \
    do {                                                                                               \
        if (dbg) {                                                                                     \
            if (per_key) SAGE_V(DD, true, true, false);                                             \
            else SAGE_V(DD, false, true, false);                                                    \
        } else if (pipe && pipe_keys) launch_pipe_i8_keys(dev->stream, p, DD, c, nw);                  \
        else if (per_key) SAGE_V(DD, true, false, true);                                            \
        else if (pipe) launch_pipe_i8(dev->stream, p, DD, c, nw);                                      \
        else SAGE_V(DD, false, false, true);                                                        \
    } while (0)
#define SAGE_F(DD, PK)                                                                                 \
    do {                                                                                               \
        if (f32o) launch_attn<DD, MODE_FP8, PK, true, false, true>(dev->stream, p, c, hm);          \
        else launch_attn<DD, MODE_FP8, PK, false, false, true>(dev->stream, p, c, hm);              \
    } while (0)
    if (fp8 && pipe) {
        if (pipe_keys) launch_pipe_fp8_keys(dev->stream, p, (int)D, c, nw);
        else launch_pipe_fp8(dev->stream, p, (int)D, c, nw);
    } else if (fp8) {
        if (D == 64) { if (per_key) SAGE_F(64, true); else SAGE_F(64, false); }
        else { if (per_key) SAGE_F(128, true); else SAGE_F(128, false); }
    } else if (D == 64) SAGE_D(64);
    else SAGE_D(128);
#undef SAGE_F
#undef SAGE_D
#undef SAGE_V
    arhip_note_selected(ARHIP_K_SAGE);
    return t.end();
}

// Q quantised inside the attention kernel (as the reference does, src/runtime/cuda_flash_sage.rs:201-223): the
// pipelined int8 (FP8) kernel with bf16 queries, scales over blocks of 128 queries.
static int sage_fwd_qfused_impl(const char *who, bool fp8, arhip_device *dev, const uint16_t *q, const int8_t *k8, const float *sk,
                               const uint16_t *v, void *o, float *sq_out, int8_t *q8_out, const int32_t *kv_len,
                               int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D, int64_t bk,
                               int causal, int out_dtype, float scale, int wait, double *secs)
{
    if (int rc = check_common(who, dev, q, k8, v, o, nullptr, B, Hq, Hkv, N, D)) return rc;
    ARHIP_REQUIRE(sk, "%s: null scale pointer", who);
    ARHIP_REQUIRE(out_dtype == ARHIP_F32 || out_dtype == ARHIP_BF16, "%s: out_dtype %d", who, out_dtype);
    int shift = 0;
    while (((int64_t)64 << shift) < bk) ++shift;
    ARHIP_REQUIRE(((int64_t)64 << shift) == bk, "%s: K scales over whole 64-key tiles (bk = 64 * 2^j), got bk = %lld", who,
                  (long long)bk);
    ARHIP_REQUIRE(pipe_addressable(N, D, 2), "%s: (N + 320) * D * 2 must stay below 2^31 (N = %lld)", who, (long long)N);
    ARHIP_REQUIRE(q8_out == nullptr || arhip_aligned16(q8_out), "%s: q8_out must be 16-byte aligned", who);
    ARHIP_HIP(hipSetDevice(dev->ordinal));
    AttnParams p = {};
    p.q = q; p.k = k8; p.v = v; p.o = o;
    p.kv_len = kv_len;
    p.sk = sk;
    p.sq_out = sq_out; p.q8_out = q8_out;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.N = (int)N;
    dense_strides(p.qs, Hq, N, D);
    dense_strides(p.ks, Hkv, N, D);
    dense_strides(p.vs, Hkv, N, D);
    dense_strides(p.os, Hq, N, D);
    p.bq = 128; p.bk = (int)bk;
    p.bk_tile_shift = shift;
    p.bk_key_shift = -1;
    p.scale = scale;
    const bool c = causal != 0;
    p.out_f32 = out_dtype == ARHIP_F32;
    const int nw = pipe_form(dev, B * Hq, N, D, false, c, kv_len != nullptr, true, D);
    p.nq = (int)((N + pipe_rows(nw) - 1) / pipe_rows(nw));
    p.total = (int)(p.nq * B * Hq);
    p.lpt = p.total <= 16 * dev->cus;
    arhip_call_timer t{dev, wait, secs};
    t.kernel = ARHIP_K_SAGE;
    if (int rc = t.begin()) return rc;
    if (fp8) launch_pipe_fp8_qf(dev->stream, p, (int)D, c, nw);
    else launch_pipe_i8_qf(dev->stream, p, (int)D, c, nw);
    arhip_note_selected(ARHIP_K_SAGE);
    return t.end();
}

extern "C" int arhip_sage_fwd_qfused(arhip_device *dev, const uint16_t *q, const int8_t *k8, const float *sk,
                                     const uint16_t *v, void *o, float *sq_out, int8_t *q8_out, const int32_t *kv_len,
                                     int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D, int64_t bk,
                                     int causal, int out_dtype, float scale, int wait, double *secs)
{
    return sage_fwd_qfused_impl("arhip_sage_fwd_qfused", false, dev, q, k8, sk, v, o, sq_out, q8_out, kv_len, B, Hq, Hkv, N, D, bk,
                                causal, out_dtype, scale, wait, secs);
}

// The same on E4M3 codes (k8 from arhip_sage_quant_fp8; the kernel derives E4M3 codes of Q with scale = absmax / 448).
extern "C" int arhip_sage_fwd_fp8_qfused(arhip_device *dev, const uint16_t *q, const uint8_t *k8, const float *sk,
                                         const uint16_t *v, void *o, float *sq_out, uint8_t *q8_out, const int32_t *kv_len,
                                         int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D, int64_t bk,
                                         int causal, int out_dtype, float scale, int wait, double *secs)
{
    return sage_fwd_qfused_impl("arhip_sage_fwd_fp8_qfused", true, dev, q, (const int8_t *)k8, sk, v, o, sq_out, (int8_t *)q8_out,
                                kv_len, B, Hq, Hkv, N, D, bk, causal, out_dtype, scale, wait, secs);
}

// The reference's own convention in one attention launch: f32 queries quantised row by row inside the kernel
// (src/runtime/cuda_flash_sage.rs:201-223), K scales per key (or per power of two of keys below 64).
extern "C" int arhip_sage_fwd_qfused_rows(arhip_device *dev, const float *q, const int8_t *k8, const float *sk,
                                          const uint16_t *v, void *o, float *sq_out, int8_t *q8_out, const int32_t *kv_len,
                                          int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D, int64_t bk,
                                          int causal, int out_dtype, float scale, int wait, double *secs)
{
    if (int rc = check_common("arhip_sage_fwd_qfused_rows", dev, q, k8, v, o, nullptr, B, Hq, Hkv, N, D)) return rc;
    ARHIP_REQUIRE(sk, "arhip_sage_fwd_qfused_rows: null scale pointer");
    ARHIP_REQUIRE(out_dtype == ARHIP_F32 || out_dtype == ARHIP_BF16, "arhip_sage_fwd_qfused_rows: out_dtype %d", out_dtype);
    int key_shift = 0;
    while (((int64_t)1 << key_shift) < bk) ++key_shift;
    ARHIP_REQUIRE(bk >= 1 && bk < 64 && ((int64_t)1 << key_shift) == bk,
                  "arhip_sage_fwd_qfused_rows: K scales over a power of two of keys below 64 (bk = 1 ... 32), got bk = %lld", (long long)bk);
    ARHIP_REQUIRE(pipe_addressable(N, D, 2), "arhip_sage_fwd_qfused_rows: (N + 320) * D * 2 must stay below 2^31 (N = %lld)", (long long)N);
    ARHIP_REQUIRE(q8_out == nullptr || arhip_aligned16(q8_out), "arhip_sage_fwd_qfused_rows: q8_out must be 16-byte aligned");
    ARHIP_HIP(hipSetDevice(dev->ordinal));
    AttnParams p = {};
    p.q = q; p.k = k8; p.v = v; p.o = o;
    p.kv_len = kv_len;
    p.sk = sk;
    p.sq_out = sq_out; p.q8_out = q8_out;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.N = (int)N;
    dense_strides(p.qs, Hq, N, D);
    dense_strides(p.ks, Hkv, N, D);
    dense_strides(p.vs, Hkv, N, D);
    dense_strides(p.os, Hq, N, D);
    p.bq = 1; p.bk = (int)bk;
    p.bk_tile_shift = 0;
    p.bk_key_shift = key_shift;
    p.scale = scale;
    const bool c = causal != 0;
    p.out_f32 = out_dtype == ARHIP_F32;
    const int nw = pipe_wants_4_waves(dev, B * Hq, N, D, c, kv_len != nullptr) ? 4 : 8;
    p.nq = (int)((N + nw * 32 - 1) / (nw * 32));
    p.total = (int)(p.nq * B * Hq);
    p.lpt = p.total <= 16 * dev->cus;
    arhip_call_timer t{dev, wait, secs};
    t.kernel = ARHIP_K_SAGE;
    if (int rc = t.begin()) return rc;
    launch_pipe_i8_keys_qf(dev->stream, p, (int)D, c, nw);
    arhip_note_selected(ARHIP_K_SAGE);
    return t.end();
}

extern "C" int arhip_sage_fwd_strided(arhip_device *dev, const int8_t *q8, const int8_t *k8,
                                      const float *sq, const float *sk, const uint16_t *v, void *o,
                                      const int64_t v_strides[3], const int64_t o_strides[3],
                                      const float *mask, const int32_t *kv_len,
                                      int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                                      int64_t bq, int64_t bk, int causal, int out_dtype, float scale,
                                      int32_t *dbg_logits, const int32_t dbg_sel[3], int wait, double *secs)
{
    return sage_fwd_impl(dev, q8, k8, sq, sk, v, o, v_strides, o_strides, mask, kv_len, B, Hq, Hkv, N, D, bq, bk, causal,
                         out_dtype, scale, dbg_logits, dbg_sel, wait, secs, false);
}

extern "C" int arhip_sage_fwd_fp8(arhip_device *dev, const uint8_t *q8, const uint8_t *k8,
                                  const float *sq, const float *sk, const uint16_t *v, void *o,
                                  const float *mask, const int32_t *kv_len,
                                  int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                                  int64_t bq, int64_t bk, int causal, int out_dtype, float scale,
                                  int wait, double *secs)
{
    return sage_fwd_impl(dev, (const int8_t *)q8, (const int8_t *)k8, sq, sk, v, o, nullptr, nullptr, mask, kv_len, B, Hq, Hkv,
                         N, D, bq, bk, causal, out_dtype, scale, nullptr, nullptr, wait, secs, true);
}

// Rows per workgroup of the backward where several query heads share a K/V head.  A dK/dV workgroup has the tiles of all of them to go
// through, and there are fewer such workgroups, so with 128 keys each long chains are left on a few compute units; 32 keys, with the
// tiles dealt out between four waves, have a chain of a quarter and four times the workgroups, at 1.6 times the time per tile.  dQ keeps 128 rows.  In
// us: what the longest chain takes, and what all workgroups take on all compute units (one at a time, and the last ones alone where
// there is not work for two rounds); 32 keys are taken where they are ahead by more than the estimate is wrong by.
// Whole backward, 128 keys / 32: D64 B5 H4/1 N1930 478 / 305, causal 447 / 183, B2 H16/4 N1024 231 / 134, causal 216 / 88, B1 H32/8 N512 113 / 50, B2
// H32/8 N200 58 / 28, B4 H24/6 N70 25 / 18, B12 H16/4 N86 27 / 23, B2 H64/8 N610 causal 283 / 139, B3 H20/10 N188 27 / 32, B2 H40/10 N2048
// 863 / 1190; D128 B2 H16/4 N1024 299 / 233, causal 295 / 155, B1 H32/8 N512 152 / 89, B8 H8/2 N512 163 / 133, B2 H8/2 N1200 331 / 187, B3 H24/6
// N700 231 / 276, causal 219 / 177, B12 H32/8 N170 136 / 169.
// Short heads, 32 keys beside 128: D128 B7 H40/10 N64 causal 64 / 57, B12 H24/6 N16 22 / 21.  (600 shapes with 2, 4 and 8 heads to a K/V head, D64
// and 128: 17 % less in the mean, and none that loses more than 2 %; without the factor 18 % and seven that lose up to 24 %.)
static BwdForm bwd_shared_form(int64_t kv_heads, int64_t group, int64_t N, int64_t D, bool causal, int cus)
{
    const int64_t t32 = (N + 31) / 32, t128 = (N + 127) / 128, q128 = kv_heads * group * t128, kv128 = kv_heads * t128, kv32 = kv_heads * t32;
    const double steps = (double)(group * t32);
    if (steps <= 2) return BWD_128;
    // of the tiles that a workgroup goes through without the causal mask
    const double of32 = causal ? 0.5 + 0.5 / t32 : 1.0, of128 = causal ? 0.5 + 0.5 / t128 : 1.0;
    // workgroups of dK/dV that take kv each in the mean, `chain` the longest, and of dQ, one on a compute unit
    auto alone = [&](int64_t n_kv, double kv, double chain, double q) {
        const double full = (double)(n_kv + q128) / cus;
        return std::max(chain, full > 1 ? ((double)n_kv * kv + (double)q128 * q) / cus + std::max(0.0, 2 - full) * q : q);
    };
    double by128, by32;
    if (D == 64) {
        const double pairs = (double)(kv_heads * group) * (double)(t32 * t32) * of128;
        by128 = std::max(8 + 1.7 * (kv128 + q128 > cus ? 1.1 : 1.0) * steps, 2.6e-3 * pairs + 10);
        by32 = alone(kv32, 8.5 + 0.55 * steps * of32, 8.5 + 0.55 * steps, 6 + 1.7 * t32 * of128);
    } else {
        // (the row scalar: a third tensor for 128 keys on short heads, a launch of 5 us else)
        const bool own_d = group * N <= 512;
        const double step = own_d ? 2.7 : 2.15;
        by128 = alone(kv128, 13 + step * steps * of128, 13 + step * steps, (own_d ? 15 : 13) + 2.2 * t32 * of128) + (own_d ? 0 : 5);
        by32 = alone(kv32, 14 + 1.1 * steps * of32, 14 + 1.1 * steps, 11 + 2.4 * t32 * of128) + 5;
    }
    return by32 < 0.88 * by128 ? BWD_128_32 : BWD_128;
}

extern "C" int arhip_flash_bwd(arhip_device *dev, const float *q, const float *k, const float *v, const float *o,
                               const float *lse, const float *dout, float *dq, float *dk, float *dv, float *delta,
                               const float *mask, const int32_t *kv_len,
                               int64_t B, int64_t Hq, int64_t Hkv, int64_t N, int64_t D,
                               int causal, float scale, int wait, double *secs)
{
    if (int rc = check_common("arhip_flash_bwd", dev, q, k, v, o, mask, B, Hq, Hkv, N, D)) return rc;
    ARHIP_REQUIRE(lse && dout && dq && dk && dv && delta, "arhip_flash_bwd: null tensor pointer");
    ARHIP_REQUIRE(arhip_aligned16(dout) && arhip_aligned16(dq) && arhip_aligned16(dk) && arhip_aligned16(dv),
                  "arhip_flash_bwd: dout/dq/dk/dv must be 16-byte aligned");
    ARHIP_REQUIRE(((reinterpret_cast<uintptr_t>(lse) | reinterpret_cast<uintptr_t>(delta)) & 3u) == 0,
                  "arhip_flash_bwd: lse/delta must be 4-byte aligned");
    ARHIP_HIP(hipSetDevice(dev->ordinal));
    arhip_call_timer t{dev, wait, secs};
    t.kernel = ARHIP_K_FLASH_BWD;
    FlashBwdParams p = {};
    p.q = q; p.k = k; p.v = v; p.dout = dout; p.lse = lse; p.delta = delta; p.mask = mask; p.kv_len = kv_len;
    p.dq = dq; p.dk = dk; p.dv = dv;
    p.Hq = (int)Hq; p.Hkv = (int)Hkv; p.N = (int)N;
    p.scale = scale;
    if (int rc = t.begin()) return rc;
    const long rows = (long)(B * Hq * N);
    // 4 waves per workgroup: 128 queries / keys that share their tiles, two workgroups on a compute unit (head size 64), or the same 32
    // queries / keys with the tiles of the other side dealt out between the waves, one on a compute unit: where all of those run at
    // once, or long heads leave the others' chains of tiles to wait for.  us, 128 / 32 rows: H8 N200 19 / 14, N512 34 / 20, H24 N200
    // (336 workgroups of 32 rows) 20 / 22, H16 N512 (512) 35 / 32, H8 N1200 (608) 63 / 76, causal H8 N1200 60 / 49, H24 N300 (480) 25 / 23,
    // H32 N300 (640) 25 / 30, H16 N800 (800) 45 / 49; a single tile, H8 N32 9.5 / 10.4.
    // Head size 128, one workgroup on a compute unit either way: H24 N64 (96) 14.5 / 18.2, H24 N128 (192) 23 / 19, H12 N197 (168) 30 / 25, H24
    // N197 (336) 30 / 36, H12 N300 (240) 37 / 28, H4 N512 (128) 54 / 32, H12 N512 (384) 57 / 54, H4 N800 (200) 75 / 47, H12 N800 (600) 79 / 110, H4
    // N1200 (304) 101 / 88, causal H24 N197 30 / 31, H12 N512 49 / 40, H12 N800 69 / 70, H4 N1200 94 / 58, H4 N2048 (512) 169 / 99, H12 N1200
    // (912) 98 / 119.
    const int64_t wgs = B * Hkv * ((N + 127) / 128), tiles32 = (N + 31) / 32, wgs32 = B * (Hq + Hkv) * tiles32;
    const int64_t cus = dev->cus;
    const bool split = D == 128 ? N > 96 && wgs32 * 2 <= cus * (causal ? (N >= 2048 ? 4 : N >= 512 ? 3 : 2) : N >= 1200 ? 3 : 2)
                       : causal ? N > 32 && (wgs32 <= cus || (N >= 256 && wgs32 * (tiles32 + 1) * 5 <= cus * tiles32 * 12))
                                : N > 32 && wgs32 <= cus * (N >= 512 ? 2 : 1);
    const BwdForm form = split ? BWD_32 : Hq == Hkv ? BWD_128 : bwd_shared_form(B * Hkv, Hq / Hkv, N, D, causal != 0, dev->cus);
    auto tiles = [&](int rows_wg) { return (int)((N + rows_wg - 1) / rows_wg); };
    p.nt_q = tiles(form == BWD_32 ? 32 : 128);
    p.nt_kv = tiles(form == BWD_128 ? 128 : 32);
    // causal: longest tile first over all heads, so that no head's long tiles are left for the end
    // Sums of dK and dV in two halves on grids of fewer than two workgroups per compute unit (as f32_tile_sums).
    p.halves = wgs < 2 * (int64_t)dev->cus;
    p.total_q = (int)(p.nt_q * B * Hq);
    p.total_kv = (int)(p.nt_kv * B * Hkv);
    // Head size 64, 128 rows: two workgroups fit a compute unit, and where there are more of them than that, but no more than three, the last dQ ones
    // begin where the first ones end, alone with a dK/dV one that has as long to go: the sooner the first ones are done the better.  us,
    // without / with priority: B8 H6 N789 (672 workgroups) 110 / 99, N700 (576) 92 / 86, B7 H12 N400 (672) 58 / 54, B8 H8 N700 (768) 112 / 103; B6 H10
    // N789 (840) 128 / 133, B12 H12 N300 (864) 57 / 61, B4 H16 N512 (512) 55 / 59, causal B8 H6 N789 (longest first) 60 / 65.
    const int64_t all = p.total_q + p.total_kv;
    p.dq_ahead = D == 64 && form == BWD_128 && !causal && all > 2 * cus && all <= 3 * cus;
    p.lpt_q = causal ? (int)(B * Hq) : 0;
    p.lpt_kv = causal ? (int)(B * Hkv) : 0;
    // The row scalar: formed by the same launch on short heads, by one before it else.  The rule goes by the queries whose tiles a key
    // tile's workgroup reads.  us, a launch of its own / the same launch: B1 H12 N197 D64 18.5 / 15.2, B4 H16 N197 27.5 / 24.6, B8 H12 N197
    // 32.4 / 31.6, B2 H16 N512 44.3 / 43.0, B8 H6 N789 113.5 / 114.6, D128 B1 H12 N197 33.9 / 32.0, B2 H16 N512 71.8 / 70.9, B8 H6 N789
    // 206 / 212, B8 H16 N1024 771 / 811; four heads to a K/V head, B8 H24 N197 60.7 / 60.9, B3 H8 N1000 causal 183 / 193.
    // (O may lie where a result or the row scalar goes: then it has to be read before they are written)
    const uintptr_t q_bytes = (uintptr_t)rows * D * 4, kv_bytes = (uintptr_t)(B * Hkv * N) * D * 4;
    auto apart = [](const void *x, uintptr_t x_bytes, const void *y, uintptr_t y_bytes) {
        const uintptr_t a = (uintptr_t)x, b = (uintptr_t)y;
        return a + x_bytes <= b || b + y_bytes <= a;
    };
    // (Head size 128 on 32 rows per workgroup has no registers for a third tensor.)
    const bool own_d = mask == nullptr && !(D == 128 && form != BWD_128) && Hq / Hkv * N <= 512 && apart(o, q_bytes, dq, q_bytes) && apart(o, q_bytes, dk, kv_bytes) &&
                       apart(o, q_bytes, dv, kv_bytes) && apart(o, q_bytes, delta, (uintptr_t)rows * 4);
    if (own_d) {
        p.o = o;
        p.delta_out = delta;
    } else {
        const int prep_rows = D == 64 ? bwd_prep_rows<64>() : bwd_prep_rows<128>();
        const dim3 prep_grid((unsigned)((rows + prep_rows - 1) / prep_rows)), block(256);
        if (D == 64) hipLaunchKernelGGL((bwd_prep_kernel<64>), prep_grid, block, 0, dev->stream, o, dout, delta, rows);
        else hipLaunchKernelGGL((bwd_prep_kernel<128>), prep_grid, block, 0, dev->stream, o, dout, delta, rows);
    }
    auto launch = [&]() {
        if (mask != nullptr) launch_f32_bwd_mask(dev->stream, p, (int)D, causal != 0, form);
        else if (D == 64) launch_f32_bwd_64(dev->stream, p, causal != 0, form);
        else launch_f32_bwd_128(dev->stream, p, causal != 0, form);
    };
    // dK and dV may lie where K and V do, of which a dK/dV workgroup reads the rows that it writes; those of dQ read all of them, first
    bool kv_kept = true;
    for (const float *out : {dk, dv})
        for (const float *in : {k, v}) kv_kept &= apart(out, kv_bytes, in, kv_bytes);
    if (kv_kept) {
        launch();
    } else {
        const int total_kv = p.total_kv;
        p.total_kv = 0;
        launch();
        p.total_kv = total_kv;
        p.total_q = 0;
        launch();
    }
    arhip_note_selected(ARHIP_K_FLASH_BWD);
    return t.end();
}
