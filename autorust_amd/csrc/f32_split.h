// fp32 contractions on the bf16 matrix instruction, at fp32 precision.
//
// (The method: G. Henry, P. T. P. Tang and A. Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations", IEEE ARITH 2019.)
//
// An fp32 value is the exact sum of three bf16 values: x = hi + mid + lo with hi = bf16(x), mid = bf16(x - hi),
// lo = x - hi - mid (24 significant bits = 3 x 8; both differences are exact, and the last one fits bf16).  A
// product a b is then the sum of nine bf16 products, each exact in the fp32 accumulator of
// v_mfma_f32_32x32x16_bf16.  The six with the largest weights are kept,
//     hi hi + (hi mid + mid hi) + (mid mid + hi lo + lo hi),
// and the three left out (mid lo, lo mid, lo lo) are at most 2^-23 of the product and about 2^-26.5 in the root
// mean square: less than the rounding of one fp32 product (2^-25.3).
//
// Six bf16 instructions contract 16 channels in 6 x 8 passes where v_mfma_f32_32x32x2_f32 takes 8 x 16, and they
// run beside the vector ALU, which the fp32 instruction does not: a matrix pipe of 2.7 times the fp32 rate that
// hides the softmax.  Rounding, measured against the exact sum: a sum of 16 products from zero on N(0,1) operands is off by 0.19
// (root mean square, in units of 2^-24 of the sum of magnitudes) per bf16 instruction, 2 products by 0.40 per fp32 one; but where
// the accumulator is much larger than the products, by 0.41 units in its last place per bf16 instruction and 0.29 per fp32 one.
// A long sum over 32-row tiles is rounded 12 times a tile here and 16 times there: variances of 2.0 and 1.3.
// Subnormal operands are multiplied as such.
//
// The three parts exist where hi does not round to infinity (|x| < 3.3962e38) and lo needs no bit below the smallest bf16
// (|x| > 2^-110, or 0).  Beyond the upper end lo (and for an infinity mid) is NaN, and so is every sum that the value enters.  Below
// the lower end up to 2^-134 of the value is lost, which counts where the other operand is huge or the sum itself that small.  A
// workgroup whose own rows (Q; dO; K, V in dK/dV) are out of range (beyond_split), or with results that are not finite or that small
// (ResultRange), therefore forms its results again with v_mfma_f32_32x32x2_f32, which multiplies operands as they are.  Looking
// at every staged value instead cost 1 % (forward) to 4 % (backward) of the time.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "attn_fwd.h"

namespace arhip {

// 8 consecutive elements of an operand row as the three parts of the matrix operand of one lane
struct split8 {
    uint4 hi, mid, lo;
};

struct split4 {  // the same of 4 elements
    uint2 hi, mid, lo;
};

// First (hi) or second (mid, lo) step of splitting a pair; a and b are left with the residuals.  The empty assembly keeps
// the packed pair as the source of both unpacked values (the compiler would convert the low one a second time).
__device__ __forceinline__ void split_take(float &a, float &b, uint32_t &part)
{
    part = pack_bf16x2(a, b);
    asm("" : "+v"(part));
    a -= __uint_as_float(part << 16);
    b -= __uint_as_float(part & 0xffff0000u);
}

__device__ __forceinline__ void split_pair(float a, float b, uint32_t &hi, uint32_t &mid, uint32_t &lo)
{
    split_take(a, b, hi);
    split_take(a, b, mid);
    lo = pack_bf16x2(a, b);
}

// Values that are computed here and nowhere later: the compiler must not sink them past this point, towards a use beyond
// the matrix instructions they are meant to run beside.
__device__ __forceinline__ void pin(float &a, float &b) { asm volatile("" : "+v"(a), "+v"(b)); }

__device__ __forceinline__ split8 split_8(float x0, float x1, float x2, float x3, float x4, float x5, float x6, float x7)
{
    split8 s;
    split_pair(x0, x1, s.hi.x, s.mid.x, s.lo.x);
    split_pair(x2, x3, s.hi.y, s.mid.y, s.lo.y);
    split_pair(x4, x5, s.hi.z, s.mid.z, s.lo.z);
    split_pair(x6, x7, s.hi.w, s.mid.w, s.lo.w);
    return s;
}

__device__ __forceinline__ split8 split_8(const float4 &a, const float4 &b)
{
    return split_8(a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w);
}

// Whether rows that a wave (or four of them) holds have a nonzero value up to 2^-110, or one from 2^100 on; a scalar.  A bf16
// code c, sign dropped and one subtracted (2 c - 1 in 16 bits), puts zero above everything else, so that a running minimum finds
// the smallest nonzero value.  Called where the wave waits for memory anyway.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
template <int STEPS>
__device__ __forceinline__ bool beyond_split(const split8 *rows)
{
    u16x2 least = {0xffff, 0xffff}, most = {0, 0};
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        const uint32_t hi[4] = {rows[i].hi.x, rows[i].hi.y, rows[i].hi.z, rows[i].hi.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, hi[j]) * (uint16_t)2 - (uint16_t)1);
            most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, hi[j] & 0x7fff7fffu));
        }
    }
    return __any(min(least.x, least.y) <= 2 * ((127 - 110) << 7) - 1 || max(most.x, most.y) >= (127 + 100) << 7);
}

// The range of results: 0 * x is NaN where x is not finite, and the bits of |x| less one put zero above everything else.
struct ResultRange {
    float mark = 0.f;
    uint32_t least = 0xffffffffu;
    __device__ __forceinline__ void take(const f32x16 &x)
    {
        float m[4] = {mark, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            m[r & 3] = fmaf(x[r], 0.f, m[r & 3]);
            least = min(least, (__float_as_uint(x[r]) << 1) - 1u);
        }
        mark = (m[0] + m[1]) + (m[2] + m[3]);
    }
    __device__ __forceinline__ void take(const float4 &x) { take(x.x); take(x.y); take(x.z); take(x.w); }
    __device__ __forceinline__ void take(float x)
    {
        mark = fmaf(x, 0.f, mark);
        least = min(least, (__float_as_uint(x) << 1) - 1u);
    }
    // not finite, or nonzero and below 2^EXP
    template <int EXP>
    __device__ __forceinline__ bool beyond() const { return mark != 0.f || least < ((uint32_t)(127 + EXP) << 24); }
};

// Whether any wave of the workgroup has something to say; flags: a word per wave, written before and read behind a barrier
__device__ __forceinline__ void flag_write(uint32_t *flags, int wave, bool mine)
{
    const bool any = __any(mine);
    if ((threadIdx.x & 63) == 0) flags[wave] = any;
}
template <int WAVES>
__device__ __forceinline__ bool flag_read(const uint32_t *flags)
{
    uint32_t any = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) any |= flags[w];
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

// For the code behind a flag: the lane and a row number that the compiler works out there, instead of keeping what depends on them in
// registers all through the tile loop.
__device__ __forceinline__ int fresh_lane() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
__device__ __forceinline__ int fresh(int scalar)
{
    asm volatile("" : "+s"(scalar));
    return scalar;
}

// c += a . b over 8 channels on the fp32 instruction; lane: row (column) lane % 32, channels 4 (lane / 32) + 0 .. 3
__device__ __forceinline__ f32x16 mfma_plain(const float4 &a, const float4 &b, f32x16 c)
{
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, c, 0, 0, 0);
}

// step 0 .. 5 of c += a . b over 16 channels (32 x 32 result), smallest products first
template <int STEP>
__device__ __forceinline__ f32x16 mfma_split_step(const split8 &a, const split8 &b, f32x16 c)
{
    const uint4 &x = STEP == 0 ? a.lo : (STEP == 2 || STEP == 3) ? a.mid : a.hi;
    const uint4 &y = STEP == 1 ? b.lo : (STEP == 2 || STEP == 4) ? b.mid : b.hi;
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 mfma_split(const split8 &a, const split8 &b, f32x16 c)
{
    c = mfma_split_step<0>(a, b, c);
    c = mfma_split_step<1>(a, b, c);
    c = mfma_split_step<2>(a, b, c);
    c = mfma_split_step<3>(a, b, c);
    c = mfma_split_step<4>(a, b, c);
    return mfma_split_step<5>(a, b, c);
}

// ---- a tile of 32 rows x D channels in LDS: three parts, each [D / 32 pieces][32 rows][64 B], the four 16-byte
// chunks of a row permuted with chunk ^= (row / 4) % 4, so that both the row reads (ds_read_b128) and the
// transposing reads (ds_read_b64_tr_b16) of 16 lanes hit 16 different 16-byte bank groups, without padding ----
template <int D>
struct SplitTile {
    static constexpr int PART = 32 * D * 2;
    static constexpr int BYTES = 3 * PART;
    // 8-channel items of a tile, in the order the staging threads take them: four chunks of a row, 32 rows, the
    // next piece (16 lanes write 256 consecutive bytes)
    static constexpr int ITEMS = 32 * D / 8;
    static __device__ __forceinline__ int item_row(int it) { return (it >> 2) & 31; }
    static __device__ __forceinline__ int item_col(int it) { return (it >> 7) * 32 + (it & 3) * 8; }  // first channel
    static __device__ __forceinline__ int item_addr(int it)
    {
        const int row = (it >> 2) & 31, c = it & 3;
        return (it >> 7) * 2048 + row * 64 + ((c ^ ((row >> 2) & 3)) * 16);
    }
    static __device__ __forceinline__ void put(unsigned char *tile, int addr, const split8 &s)
    {
        *(uint4 *)(tile + addr) = s.hi;
        *(uint4 *)(tile + PART + addr) = s.mid;
        *(uint4 *)(tile + 2 * PART + addr) = s.lo;
    }
    static __device__ __forceinline__ void put(unsigned char *tile, int addr, const split4 &s)
    {
        *(uint2 *)(tile + addr) = s.hi;
        *(uint2 *)(tile + PART + addr) = s.mid;
        *(uint2 *)(tile + 2 * PART + addr) = s.lo;
    }
    // operand rows: lane = row i32, channels 16 st + 8 h .. + 7.  addr = row_addr(lane, st & 1) + (st / 2) * 2048
    static __device__ __forceinline__ int row_addr(int i32, int h, int odd)
    {
        return i32 * 64 + (((2 * odd + h) ^ ((i32 >> 2) & 3)) * 16);
    }
    template <int P>  // part 0 hi, 1 mid, 2 lo
    static __device__ __forceinline__ uint4 get_row_part(const unsigned char *tile, int addr)
    {
        return *(const uint4 *)(tile + P * PART + addr);
    }
    static __device__ __forceinline__ split8 get_row(const unsigned char *tile, int addr)
    {
        return {get_row_part<0>(tile, addr), get_row_part<1>(tile, addr), get_row_part<2>(tile, addr)};
    }
    // operand columns (the transposed tile): lane = channel 32 db + i32, rows 16 ks + 4 h + {0..3} and
    // 16 ks + 8 + 4 h + {0..3}, the rows whose values a result of the 32 x 32 instruction leaves in registers
    // 8 ks .. 8 ks + 7.  addr = col_addr(lane, second) + db * 2048 + ks * 1024
    static __device__ __forceinline__ int col_addr(int lane, int second)
    {
        const int h = lane >> 5, r = 4 * h + ((lane & 15) >> 2) + 8 * second;
        const int c = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
        return r * 64 + ((c ^ ((r >> 2) & 3)) * 16) + (lane & 1) * 8;
    }
    template <int P>
    static __device__ __forceinline__ uint4 get_col_part(const unsigned char *tile, int a0, int a1)
    {
        const uint2 x = lds_read_tr16(tile + P * PART + a0), y = lds_read_tr16(tile + P * PART + a1);
        return make_uint4(x.x, x.y, y.x, y.y);
    }
    static __device__ __forceinline__ split8 get_col(const unsigned char *tile, int a0, int a1)
    {
        return {get_col_part<0>(tile, a0, a1), get_col_part<1>(tile, a0, a1), get_col_part<2>(tile, a0, a1)};
    }
};


// ---- the interleaved instruction stream ----
// The operand fragment being multiplied and, part by part as its registers fall free, the next one: the next lo part
// replaces lo behind the first of the six products, mid behind the fourth, and hi has two sets of registers.
struct SplitFrag {
    uint4 lo, mid, hi[2];
    template <int SET, int P>
    __device__ __forceinline__ void set(const uint4 &x)
    {
        if constexpr (P == 0) hi[SET] = x;
        else if constexpr (P == 1) mid = x;
        else lo = x;
    }
    template <int SET>
    __device__ __forceinline__ split8 get() const { return {hi[SET], mid, lo}; }
};

// NF fragments (an even number), six matrix instructions each, with NSTEPS vector steps dealt out between them.  A wave
// issues in order and may issue vector instructions while a matrix instruction runs; the fences keep the order as written.
//   mul(f, m)   product m of fragment f
//   load(f, P)  reads part P of fragment f (f = 1 .. NF; NF is the first one of what follows)
//   step(i)     vector work
template <int NF, int NSTEPS, typename Mul, typename Load, typename Step>
__device__ __forceinline__ void mfma_region(Mul &&mul, Load &&load, Step &&step)
{
    static_assert(NF % 2 == 0, "the fragment after the region goes to the first register set");
    static_for<0, 6 * NF>([&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, f = i / 6, m = i % 6;
        mul(std::integral_constant<int, f>{}, std::integral_constant<int, m>{});
        if constexpr (m == 0) load(std::integral_constant<int, f + 1>{}, std::integral_constant<int, 2>{});
        if constexpr (m == 1) load(std::integral_constant<int, f + 1>{}, std::integral_constant<int, 0>{});
        if constexpr (m == 3) load(std::integral_constant<int, f + 1>{}, std::integral_constant<int, 1>{});
        static_for<i * NSTEPS / (6 * NF), (i + 1) * NSTEPS / (6 * NF)>(step);
        ARHIP_FENCE();
    });
}

// Splitting 8 values into an operand (or 4, where registers are short), one operation of four pairs at a time: the four instructions of a step are
// independent of each other and of everything since the matrix instruction before last, so a wave that has its SIMD to
// itself issues them without waiting (a step that runs one pair from conversion to residual costs it twice the time:
// measured, cycles per matrix instruction with six dependent / independent vector instructions behind it: 60 / 40, with
// four 44 / 36, with two waves per SIMD 36 / 34).  x is left with the residuals; t is scratch.
constexpr int SPLIT_STEPS = 11;
template <int OP, typename S>
__device__ __forceinline__ void split_op(float *x, uint32_t *t, S &s)
{
    uint32_t *part = (uint32_t *)(OP < 5 ? &s.hi : OP < 10 ? &s.mid : &s.lo);
#pragma unroll
    for (int i = 0; i < (int)sizeof(s.hi) / 4; ++i) {
        constexpr int k = OP % 5;
        if constexpr (k == 0) {
            part[i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
            asm volatile("" : "+v"(part[i]));
        } else if constexpr (k == 1) {
            t[i] = part[i] << 16;
            asm volatile("" : "+v"(t[i]));
        } else if constexpr (k == 3) {
            t[i] = part[i] & 0xffff0000u;
            asm volatile("" : "+v"(t[i]));
        } else {
            float &v = x[2 * i + (k == 4)];
            v -= __uint_as_float(t[i]);
            asm volatile("" : "+v"(v));
        }
    }
}

}  // namespace arhip
