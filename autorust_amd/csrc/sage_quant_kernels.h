// Kernels of the Sage pre-pass: K mean (smoothing), per-block / per-row symmetric int8
// quantisation, f32 -> bf16 cast.  All of it is HBM-bound streaming work.
//
// The quantisation rule is the reference's (src/runtime/cuda_flash_sage.rs):
//   scale = absmax > 0 ? absmax / 127 : 1      (:209-213, :264-268)
//   inv   = 1 / scale                          (:218, :273)
//   x8    = clamp(rint(x * inv), -127, 127)    (:124-137), rint = nearest-even
// hoisted out of the attention kernel (the reference re-quantises K for every query block,
// :248-278) and applied to blocks of tokens instead of single rows.  Every fp32 operation is a
// single IEEE operation in a fixed order, so the int8 tensors and scales are bit-reproducible on
// the CPU.  Each kernel is a __device__ body plus a __global__ template; the loadable code
// object wraps the same bodies in named entry points.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lane_max.h"

#pragma clang fp contract(off)

namespace arhip {

constexpr int MEAN_CHUNK = 64;  // tokens per partial sum

// Where the input tensor's rows are: element strides of batch / head / token (the channel stride
// is 1).  Dense [B, H, N, D] is {H*N*D, N*D, D}; the token-major layout a projection produces,
// [B, N, H, D], is {N*H*D, D, H*D}.  Outputs of the pre-pass are always dense.
struct XLayout {
    long sb, sh, st;
    int H;
    __host__ __device__ static XLayout dense(int H, int N, int D) { return {(long)H * N * D, (long)N * D, (long)D, H}; }
    __device__ __forceinline__ size_t head(int bh) const { return (size_t)(bh / H) * sb + (size_t)(bh % H) * sh; }
};


__device__ __forceinline__ void ld8(const float *x, size_t e, float v[8])
{
    const float4 a = *(const float4 *)(x + e), b = *(const float4 *)(x + e + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void ld8(const uint16_t *x, size_t e, float v[8])
{
    const uint4 a = *(const uint4 *)(x + e);
    v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
    v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
    v[4] = __uint_as_float(a.z << 16); v[5] = __uint_as_float(a.z & 0xffff0000u);
    v[6] = __uint_as_float(a.w << 16); v[7] = __uint_as_float(a.w & 0xffff0000u);
}

// two adjacent channels
__device__ __forceinline__ void ld2(const float *x, size_t e, float v[2])
{
    const float2 a = *(const float2 *)(x + e);
    v[0] = a.x; v[1] = a.y;
}
__device__ __forceinline__ void ld2(const uint16_t *x, size_t e, float v[2])
{
    const uint32_t a = *(const uint32_t *)(x + e);
    v[0] = __uint_as_float(a << 16); v[1] = __uint_as_float(a & 0xffff0000u);
}

// s[0..C) = x[j0] + x[j0 + 1] + ... + x[j1 - 1] of C (8 or 2) adjacent channels in token order; base: the channels of token 0.
// U rows are in flight per thread (their loads are issued together) and added in token order: a short sequence has few
// threads, and its time is the number of load round trips and of instructions of a wave that has its SIMD to itself.
template <int U, int C, typename T>
__device__ __forceinline__ void sum_rows(const T *x, size_t base, long st, int j0, int j1, float (&s)[C])
{
    auto ld = [&](int j, float *v) __attribute__((always_inline)) {
        if constexpr (C == 8) ld8(x, base + (size_t)j * st, v);
        else ld2(x, base + (size_t)j * st, v);
    };
#pragma unroll
    for (int i = 0; i < C; ++i) s[i] = 0.f;
    int j = j0;
    for (; j + U <= j1; j += U) {
        float v[U][C];
#pragma unroll
        for (int u = 0; u < U; ++u) ld(j + u, v[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < C; ++i) s[i] += v[u][i];
    }
    for (; j < j1; j += 8) {  // the last row stands in for those past the end and is not added
        float v[8][C];
#pragma unroll
        for (int u = 0; u < 8; ++u) ld(min(j + u, j1 - 1), v[u]);
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (j + u < j1) {
#pragma unroll
                for (int i = 0; i < C; ++i) s[i] += v[u][i];
            }
    }
}

// part[bh][c][d] = k[64c][d] + k[64c+1][d] + ... in token order, for channels C g .. C g + C - 1
template <typename T, int C>
__device__ __forceinline__ void k_mean_chunk(const T *x, float *part, int N, int D, int nchunk, const XLayout lay, int bh, int c, int g)
{
    float s[C];
    sum_rows<(C == 8 ? 16 : 32), C>(x, lay.head(bh) + g * C, lay.st, c * MEAN_CHUNK, min(N, (c + 1) * MEAN_CHUNK), s);
    float *o = part + ((size_t)bh * nchunk + c) * D + g * C;
    if constexpr (C == 8) {
        *(float4 *)o = make_float4(s[0], s[1], s[2], s[3]);
        *(float4 *)(o + 4) = make_float4(s[4], s[5], s[6], s[7]);
    } else {
        *(float2 *)o = make_float2(s[0], s[1]);
    }
}

// One thread owns C adjacent channels of one 64-token chunk: D/C threads read a whole row
// (coalesced), 256/(D/C) chunks per workgroup.  bf16: C = 2, four times the waves of C = 8
// (by kernel trace, B4 H32 N8192 D128 56 -> 48 us, 5.6 TB/s, B2 H32 N4096 14.6 -> 11.9, B2 H32 N11403 D64 15.8 -> 15.4; with the 64 rows of a chunk
// in flight 3 % less, 8 and 9 % more, and B2 H40 N2020 D128 10.0 in place of 8.7).  f32: C = 8 for the memory's rate, 2 where the tensor
// is small and a wave's own instructions are the time (B2 Hkv8 N2016 D64: 6.0 -> 4.5 us).
template <typename T, int C>
__device__ __forceinline__ void k_mean_partial_body(const T *x, float *part, int N, int D, int nchunk, const XLayout lay, const dim3 bid)
{
    const int gpr = D / C, c = bid.x * (256 / gpr) + threadIdx.x / gpr;
    if (c < nchunk) k_mean_chunk<T, C>(x, part, N, D, nchunk, lay, bid.y, c, threadIdx.x % gpr);
}

// The grid of C = 8; a workgroup that has chunks for less than half of its threads deals them out two channels at a time.
template <typename T>
__device__ __forceinline__ void k_mean_partial_any(const T *x, float *part, int N, int D, int nchunk, const XLayout lay, const dim3 bid)
{
    const int cpb = 256 / (D / 8), c0 = bid.x * cpb, n = min(cpb, nchunk - c0), gpr = D / 2;
    if (2 * n > cpb) {
        k_mean_partial_body<T, 8>(x, part, N, D, nchunk, lay, bid);
    } else {
        for (int i = threadIdx.x; i < n * gpr; i += 256) k_mean_chunk<T, 2>(x, part, N, D, nchunk, lay, bid.y, c0 + i / gpr, i % gpr);
    }
}

template <typename T, int C>
__global__ void __launch_bounds__(256) k_mean_partial_kernel(const T *x, float *part, int N, int D, int nchunk, const XLayout lay)
{
    k_mean_partial_body<T, C>(x, part, N, D, nchunk, lay, blockIdx);
}

// (p[0] + p[D] + ...) / N: the mean of one channel from its nchunk partial sums in memory, in chunk order, on top of tot, the first c of them.
// Its time is the number of load round trips, of a kernel of few waves or at the head of a workgroup's work, and behind that the number of loads: up
// to 32 at a time, the last sum stands in for those past the end and is not added, in the smallest of four sizes that holds what is left.
// Pre-pass of f32 rows, us, with exact batches of 32, 8 and 1 / batches of 32 only / now: blocks of 64, B2 H24 N1400 D64 (22 sums) 13.7 / 12.9 / 12.5, B1
// H8 N789 D128 (13) 9.6 / 8.8 / 8.3, B3 H12 N508 D128 (8) 9.9 / 10.9 / 9.9, B2 H4 N2169 D128 (34) 10.5 / 11.0 / 10.4; rows, B2 H4 N96 D128 (2) 7.2 / 7.5 / 7.2.
__device__ __forceinline__ float mean_of_chunks(const float *p, int N, int D, int nchunk, float tot = 0.f, int c = 0)
{
    auto trip = [&](auto u) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        float v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) v[i] = p[(size_t)min(c + i, nchunk - 1) * D];
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (c + i < nchunk) tot += v[i];
        c += U;
    };
    while (nchunk - c > 16) trip(std::integral_constant<int, 32>{});
    if (nchunk - c > 8) trip(std::integral_constant<int, 16>{});
    else if (nchunk - c > 4) trip(std::integral_constant<int, 8>{});
    else if (nchunk - c > 0) trip(std::integral_constant<int, 4>{});
    return tot / (float)N;
}

// The same from all sums, in LDS: no trip to save there, and a read or a condition more is time that every workgroup waits, so exactly as many as
// there are.  Pre-pass, us, in batches of 8 of which the last one is not full / now: bf16, B1 H8 N513 D64 5.0 / 4.9, B2 H6 N577 6.4 / 6.3, B2 H4 N700
// D128 7.9 / 7.8, f32 to fp8, B4 H16 N60 D128 5.8 / 5.6.  FINE: batches of 4 and 2 in between (bf16, B1 H12 N960 D64 6.2 / 6.1, B1 H6 N300 4.7 / 4.6;
// f32 to fp8, B4 H16 N60 D128 5.6 / 5.8).
template <bool FINE>
__device__ __forceinline__ float mean_of_lds_chunks(const float *p, int N, int D, int nchunk)
{
    float tot = 0.f;
    int c = 0;
    auto batches = [&](auto u) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        for (; c + U <= nchunk; c += U) {
            float v[U];
#pragma unroll
            for (int i = 0; i < U; ++i) v[i] = p[(c + i) * D];
#pragma unroll
            for (int i = 0; i < U; ++i) tot += v[i];
        }
    };
    batches(std::integral_constant<int, 32>{});
    batches(std::integral_constant<int, 8>{});
    if constexpr (FINE) {
        batches(std::integral_constant<int, 4>{});
        batches(std::integral_constant<int, 2>{});
    }
    batches(std::integral_constant<int, 1>{});
    return tot / (float)N;
}

__device__ __forceinline__ void k_mean_final_body(const float *part, float *mean, int N, int D, int nchunk, const dim3 bid)
{
    const int bh = bid.x, d = threadIdx.x;
    mean[(size_t)bh * D + d] = mean_of_chunks(part + (size_t)bh * nchunk * D + d, N, D, nchunk);
}

// One wave or two per head: bound by the round trips to the partial sums, 1.1 us each, so 128 and 64 of them go together where there are as
// many (D by the template: their offsets are immediates; from D = 128 at run time they spill 428 scalar registers).  B1 H64 N32768 D128 (512 sums) in
// batches of 32 17.5 us, so 8.0; B4 H32 N8192 4.9 -> 4.7.
template <int D>
__global__ void __launch_bounds__(D) k_mean_final_kernel(const float *part, float *mean, int N, int nchunk)
{
    const int bh = blockIdx.x, d = threadIdx.x;
    const float *p = part + (size_t)bh * nchunk * D + d;
    float tot = 0.f;
    int c = 0;
    auto full = [&](auto u) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        float v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) v[i] = p[(size_t)c * D + i * D];
#pragma unroll
        for (int i = 0; i < U; ++i) tot += v[i];
        c += U;
    };
    while (nchunk - c >= 128) full(std::integral_constant<int, 128>{});
    if (nchunk - c >= 64) full(std::integral_constant<int, 64>{});
    mean[(size_t)bh * D + d] = mean_of_chunks(p, N, D, nchunk, tot, c);
}

// FP8 E4M3 (OCP "FN" flavour: bias 7, no infinities, largest finite 448) of the reference's AR_FP8
// branch: `__nv_cvt_float2_to_fp8x2(..., __NV_SATFINITE, __NV_E4M3)`, src/runtime/cuda_flash_sage.rs:125-128,
// with scale = absmax / 448 (:9).  The hardware conversion rounds to nearest even; the operands
// are clamped to +-448 first, which is what SATFINITE does to anything larger (values in
// (448, 464) round down to 448 either way).
template <bool FP8>
struct QFormat {
    static constexpr float QMAX = FP8 ? 448.0f : 127.0f;
};
template <bool FP8>
__device__ __forceinline__ uint2 quantise8(const float (&v)[8], float inv)
{
    uint32_t w[2] = {0u, 0u};
    if constexpr (FP8) {
        float c[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = fminf(fmaxf(v[i] * inv, -448.0f), 448.0f);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            int r = 0;
            r = __builtin_amdgcn_cvt_pk_fp8_f32(c[4 * j + 0], c[4 * j + 1], r, false);
            r = __builtin_amdgcn_cvt_pk_fp8_f32(c[4 * j + 2], c[4 * j + 3], r, true);
            w[j] = (uint32_t)r;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int iv = (int)rintf(v[i] * inv);
            iv = iv < -127 ? -127 : (iv > 127 ? 127 : iv);
            w[i >> 2] |= ((uint32_t)iv & 0xffu) << ((i & 3) * 8);
        }
    }
    return make_uint2(w[0], w[1]);
}

// One workgroup of NT threads per (block of `blk` tokens, head).  Blocks of up to 256*64 elements are kept
// in registers between the absmax pass and the quantising pass (one trip to memory); larger
// ones are read twice.  mu: the mean of this head's channels (SMOOTH).
template <typename T, bool SMOOTH, bool FP8 = false, int NT = 256>
__device__ __forceinline__ void quant_block(const T *x, int8_t *x8, float *scales, const float *mu,
                                            int N, int D, int blk, int nblk, const XLayout lay, const dim3 bid)
{
    constexpr int KEEP = 2048 / NT;  // 8-element groups a thread can hold
    __shared__ float red[NT / 64];  // one instance per kernel that inlines this body
    const int bi = bid.x, bh = bid.y, tid = threadIdx.x;
    const int r0 = bi * blk;
    const int r1 = min(N, r0 + blk);
    const size_t base = ((size_t)bh * N + r0) * D;  // of the dense output
    const size_t xbase = lay.head(bh) + (size_t)r0 * lay.st;
    // element e of the block (row e / D, channel e % D) in the input
    auto xin = [&](int e) __attribute__((always_inline)) { return xbase + (size_t)(e / D) * lay.st + (e % D); };
    const int nelem = (r1 - r0) * D;  // multiple of 8
    const bool keep = nelem <= NT * 8 * KEEP;

    float held[KEEP][8];
    float mx = 0.f;
    if (keep) {
#pragma unroll
        for (int it = 0; it < KEEP; ++it) {
            const int e = (it * NT + tid) * 8;
            if (e < nelem) {
                ld8(x, xin(e), held[it]);
                const int d = e % D;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (SMOOTH) held[it][i] = held[it][i] - mu[d + i];
                    mx = fmaxf(mx, fabsf(held[it][i]));
                }
            }
        }
    } else {
        for (int e = tid * 8; e < nelem; e += NT * 8) {
            float v[8];
            ld8(x, xin(e), v);
            const int d = e % D;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float xv = v[i];
                if (SMOOTH) xv = xv - mu[d + i];
                mx = fmaxf(mx, fabsf(xv));
            }
        }
    }
    mx = lane_group_max<64>(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) mx = fmaxf(mx, red[w]);

    const float scale = (mx > 0.f) ? mx / QFormat<FP8>::QMAX : 1.f;
    const float inv = 1.f / scale;
    if (tid == 0) scales[(size_t)bh * nblk + bi] = scale;

    auto quant8 = [&](const float (&v)[8]) { return quantise8<FP8>(v, inv); };
    if (keep) {
#pragma unroll
        for (int it = 0; it < KEEP; ++it) {
            const int e = (it * NT + tid) * 8;
            if (e < nelem) *(uint2 *)(x8 + base + e) = quant8(held[it]);
        }
    } else {
        for (int e = tid * 8; e < nelem; e += NT * 8) {
            float v[8];
            ld8(x, xin(e), v);
            const int d = e % D;
            if (SMOOTH) {
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = v[i] - mu[d + i];
            }
            *(uint2 *)(x8 + base + e) = quant8(v);
        }
    }
}

template <typename T, bool SMOOTH, bool FP8 = false>
__device__ __forceinline__ void quant_blocks_body(const T *x, int8_t *x8, float *scales, const float *mean,
                                                  int N, int D, int blk, int nblk, const XLayout lay, const dim3 bid)
{
    quant_block<T, SMOOTH, FP8>(x, x8, scales, SMOOTH ? mean + (size_t)bid.y * D : nullptr, N, D, blk, nblk, lay, bid);
}

// The smoothing quantiser with fewer launches, for sequences where a launch costs more than the work it does: every
// workgroup of a head forms the head's mean for itself, with the same sums in the same order, and the first one writes it.
// ONE: from the rows (one launch instead of three; every workgroup reads the whole head, two channels per thread).
// Otherwise from the partial sums of k_mean_partial_kernel (two launches instead of three).
// nchunk * D <= SMOOTH_LDS_FLOATS with ONE.  Pre-pass, kernel times and the gaps between them: B2 Hkv3 N374 D128 12 -> 6.5 us (ONE),
// B2 Hkv8 N2016 D64 15 -> 10 us (partial sums).
constexpr int SMOOTH_LDS_FLOATS = 2048;
template <bool ONE>
constexpr int smooth_threads() { return ONE ? 1024 : 256; }
template <typename T, bool FP8, bool ONE>
__global__ void __launch_bounds__(smooth_threads<ONE>()) smooth_quant_blocks_kernel(const T *x, int8_t *x8, float *scales, const float *part,
                                                                                  float *mean, int N, int D, int blk, int nblk, int nchunk,
                                                                                  const XLayout lay)
{
    constexpr int NT = smooth_threads<ONE>();
    __shared__ float sums[ONE ? SMOOTH_LDS_FLOATS : 1], mu[128];
    const int bh = blockIdx.y, tid = threadIdx.x;
    if constexpr (ONE) {
        const int gpr = D / 2, g = tid % gpr;
        for (int c = tid / gpr; c < nchunk; c += NT / gpr) {
            float s[2];
            sum_rows<32, 2>(x, lay.head(bh) + g * 2, lay.st, c * MEAN_CHUNK, min(N, (c + 1) * MEAN_CHUNK), s);
            *(float2 *)&sums[c * D + g * 2] = make_float2(s[0], s[1]);
        }
        __syncthreads();
    }
    if (tid < D) {
        mu[tid] = ONE ? mean_of_lds_chunks<!(FP8 && sizeof(T) == 4)>(sums + tid, N, D, nchunk) : mean_of_chunks(part + (size_t)bh * nchunk * D + tid, N, D, nchunk);
        if (blockIdx.x == 0) mean[(size_t)bh * D + tid] = mu[tid];
    }
    __syncthreads();
    quant_block<T, true, FP8, NT>(x, x8, scales, mu, N, D, blk, nblk, lay, blockIdx);
}

// The codes of 8 values that share a scale of ordinary size: quantise8 without what only matters elsewhere.  |v inv| is at most 127 (448) and
// a rounding or two, so int8 needs no clamp, and the sum with 1.5 * 2^23 is rounded to a whole number as rintf rounds, whose last byte is the
// code; a NaN's is 0, as the conversion's is, where its last bits are (every NaN that comes of bf16 values).  (v_med3_f32 takes the
// smallest of its operands where one is NaN: -448, as fmaxf does.)
template <bool FP8>
__device__ __forceinline__ uint2 quantise8_usual(const float (&v)[8], float inv)
{
    uint32_t w[2];
    if constexpr (FP8) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float c[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) c[i] = __builtin_amdgcn_fmed3f(v[4 * j + i] * inv, -448.0f, 448.0f);
            int r = 0;
            r = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], r, false);
            r = __builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], r, true);
            w[j] = (uint32_t)r;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32_t b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = __float_as_uint(v[4 * j + i] * inv + 12582912.0f);
            const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u), hi = __builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u);
            w[j] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        }
    }
    return make_uint2(w[0], w[1]);
}

// quant_blocks<uint16_t, true, FP8> for blocks of 64 tokens, the same results: 16 bytes of 4 rows per thread, so that a workgroup has one block at
// D = 128 and two at D = 64.  PART: the mean comes from the partial sums, which are read and added behind the requests of the rows (a
// launch less); else it is there.
// Bound: memory.  By kernel trace, B4 H32 N8192 D128 (402 MB, a part of which a cache holds) 84 -> 59 us, B2 H32 N4096 D128 21 -> 16, B2 H32 N11403
// D64 28 -> 21, against quant_blocks, which issues twice as many instructions per value (8 to unpack, quantise and clamp one) and at D = 64 fills its threads half.
template <int D, bool FP8, bool PART>
__global__ void __launch_bounds__(256) smooth_quant_64_kernel(const uint16_t *x, int8_t *x8, float *scales, const float *part, float *mean,
                                                              int N, int nchunk, const XLayout lay)
{
    constexpr int GPR = D / 8, TPB = 16 * GPR, BLOCKS = 256 / TPB;  // threads per row and per block, blocks per workgroup
    __shared__ float red[4], mu_of[PART ? D : 1];
    const int tid = threadIdx.x, g = tid % GPR * 8;
    // from the end: the rows that the sums were formed of last are those that a cache may still hold (B4 H32 N8192 D128 126 -> 122 us
    // for the whole pre-pass)
    const int bh = gridDim.y - 1 - blockIdx.y, c = (gridDim.x - 1 - blockIdx.x) * BLOCKS + tid / TPB;
    const int r0 = c * 64 + tid % TPB / GPR;  // the thread's first row; the others are 16 apart
    const uint16_t *src = x + lay.head(bh) + g;

    uint4 raw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) raw[i] = *(const uint4 *)(src + (size_t)min(r0 + 16 * i, N - 1) * lay.st);
    float mu[8];
    if constexpr (PART) {
        if (tid < D) {
            mu_of[tid] = mean_of_chunks(part + (size_t)bh * nchunk * D + tid, N, D, nchunk);
            if (blockIdx.x == 0) mean[(size_t)bh * D + tid] = mu_of[tid];
        }
        __syncthreads();
    }
    const float *m = PART ? mu_of + g : mean + (size_t)bh * D + g;
#pragma unroll
    for (int i = 0; i < 8; ++i) mu[i] = m[i];
    float v[4][8], mx = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[i][2 * j] = __uint_as_float(w[j] << 16) - mu[2 * j];
            v[i][2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u) - mu[2 * j + 1];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(v[i][j]));
    }
    // (rows past the end repeat the last one, which is of the same block where the block has a row at all)
    mx = lane_group_max<64>(mx);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    const int w0 = tid / TPB * (TPB / 64);
    mx = fmaxf(red[w0], red[w0 + 1]);
    if constexpr (TPB == 256) mx = fmaxf(mx, fmaxf(red[2], red[3]));
    const float scale = (mx > 0.f) ? mx / QFormat<FP8>::QMAX : 1.f;
    const float inv = 1.f / scale;
    if (c < nchunk && tid % TPB == 0) scales[(size_t)bh * nchunk + c] = scale;
    const bool usual = scale > 0x1p-100f && scale < 0x1p100f;
    int8_t *dst = x8 + (size_t)bh * N * D + g;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = r0 + 16 * i;
        const uint2 q = usual ? quantise8_usual<FP8>(v[i], inv) : quantise8<FP8>(v[i], inv);
        if (r < N) *(uint2 *)(dst + (size_t)r * D) = q;
    }
}

template <typename T, bool SMOOTH, bool FP8 = false>
__global__ void __launch_bounds__(256) quant_blocks_kernel(const T *x, int8_t *x8, float *scales, const float *mean,
                                                           int N, int D, int blk, int nblk, const XLayout lay)
{
    quant_blocks_body<T, SMOOTH, FP8>(x, x8, scales, mean, N, D, blk, nblk, lay, blockIdx);
}

// The reference's own granularity, one scale per token row (block == 1): D/8 lanes share a row,
// so a workgroup of 256 threads quantises 256/(D/8) rows and the absmax is a shuffle reduction
// inside the lane group.  Same arithmetic, same order of operations per element.
template <typename T, bool SMOOTH, bool FP8 = false>
__device__ __forceinline__ void quant_rows_body(const T *x, int8_t *x8, float *scales, const float *mean,
                                                int N, int D, long rows_total, const XLayout lay, const dim3 bid)
{
    const int gpr = D / 8;                                   // lanes per row (8 or 16)
    const long row = (long)bid.x * (256 / gpr) + threadIdx.x / gpr;   // global row over [B*H*N]
    const int g = threadIdx.x % gpr;
    const bool live = row < rows_total;
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (live) {
        ld8(x, lay.head((int)(row / N)) + (size_t)(row % N) * lay.st + g * 8, v);
        if (SMOOTH) {
            const float *mu = mean + (size_t)(row / N) * D + g * 8;
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = v[i] - mu[i];
        }
    }
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(v[i]));
    mx = gpr == 16 ? lane_group_max<16>(mx) : lane_group_max<8>(mx);
    const float scale = (mx > 0.f) ? mx / QFormat<FP8>::QMAX : 1.f;
    const float inv = 1.f / scale;
    if (live) {
        if (g == 0) scales[row] = scale;
        *(uint2 *)(x8 + (size_t)row * D + g * 8) = quantise8<FP8>(v, inv);
    }
}

template <typename T, bool SMOOTH, bool FP8 = false>
__global__ void __launch_bounds__(256) quant_rows_kernel(const T *x, int8_t *x8, float *scales, const float *mean,
                                                         int N, int D, long rows_total, const XLayout lay)
{
    quant_rows_body<T, SMOOTH, FP8>(x, x8, scales, mean, N, D, rows_total, lay, blockIdx);
}

// y[0, n) = bf16(x[0, n)), round to nearest even, by `groups` workgroups of which this is number `group`; 8 values per
// thread and step where both pointers are 16-byte aligned
__device__ __forceinline__ void cast_rows_bf16(const float *x, uint16_t *y, size_t n, size_t group, size_t groups)
{
    const size_t i0 = group * blockDim.x + threadIdx.x, stride = groups * blockDim.x;
    size_t done = 0;
    if ((((uintptr_t)x | (uintptr_t)y) & 15u) == 0) {
        for (size_t i = i0; i < n / 8; i += stride) {
            float v[8];
            ld8(x, i * 8, v);
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const __bf16 a = (__bf16)v[2 * j], b = (__bf16)v[2 * j + 1];
                w[j] = (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
            }
            *(uint4 *)(y + i * 8) = make_uint4(w[0], w[1], w[2], w[3]);
        }
        done = n / 8 * 8;
    }
    for (size_t i = done + i0; i < n; i += stride) {
        const __bf16 b = (__bf16)x[i];
        y[i] = __builtin_bit_cast(uint16_t, b);
    }
}

__device__ __forceinline__ void cast_bf16_body(const float *x, uint16_t *y, size_t n, const dim3 bid)
{
    cast_rows_bf16(x, y, n, bid.x, gridDim.x);
}

__global__ void __launch_bounds__(256) cast_bf16_kernel(const float *x, uint16_t *y, size_t n)
{
    cast_bf16_body(x, y, n, blockIdx);
}

// The reference's pre-pass for K and V in one launch (f32 tensors, a scale per key, no smoothing): workgroups
// [0, row_blocks) quantise rows of K as quant_rows does, the rest cast V to bf16 as cast_bf16 does.  Two launches of a
// few microseconds each become one; results are those of the two kernels bit for bit.
__device__ __forceinline__ void quant_rows_cast_body(const float *k, int8_t *k8, float *scales, const float *v, uint16_t *vb,
                                                     int N, int D, long rows_total, long nv, int row_blocks, const dim3 bid)
{
    if ((int)bid.x < row_blocks) {
        quant_rows_body<float, false>(k, k8, scales, nullptr, N, D, rows_total, XLayout::dense(1, N, D), bid);
    } else {
        cast_rows_bf16(v, vb, (size_t)nv, bid.x - row_blocks, gridDim.x - row_blocks);
    }
}

__global__ void __launch_bounds__(256) quant_rows_cast_kernel(const float *k, int8_t *k8, float *scales, const float *v,
                                                              uint16_t *vb, int N, int D, long rows_total, long nv, int row_blocks)
{
    quant_rows_cast_body(k, k8, scales, v, vb, N, D, rows_total, nv, row_blocks, blockIdx);
}


}  // namespace arhip
