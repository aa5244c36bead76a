// fp32 FlashAttention backward: the softmax-backward row scalar, dQ, and dK/dV.
//
// Semantics of the reference's training kernels (src/runtime/cuda_flash_train.rs:145-309):
//   prep   D[bh, i]  = sum_d O[i, d] dO[i, d]
//   dQ     s = (q_i . k_j) scale (+ mask[i, j]);  p = lse_i > -5e29 ? exp(s - lse_i) : 0;
//          dp = dO_i . v_j;  ds = p (dp - D_i) scale;  dQ_i = sum_j ds k_j
//   dK/dV  dK_j = sum_{g, i} ds q_i;  dV_j = sum_{g, i} p dO_i   (g over the GQA group of the K/V head,
//          in a fixed order: no atomics, bit-reproducible)
// Keys past the diagonal (causal) or past kv_len contribute p = 0.  head_dim and scale are parameters
// here (the reference hard-codes 64 and 0.125).
//
// All contractions run on the bf16 matrix instruction with every fp32 operand as the exact sum of three bf16 values
// (f32_split.h), with the decomposition of the forward kernel (flash_f32.h): one row of the "resident" operand per lane.
//   dQ kernel   a wave owns 32 queries (lane = query): S^T = K Q^T and dP^T = V dO^T leave, per lane,
//               16 keys of one query, so lse_i and D_i are per-lane scalars and dS^T is already the B
//               operand of dQ^T += K^T dS^T.  K and V tiles of 32 keys are staged in LDS.
//   dK/dV kernel  a wave owns 32 keys (lane = key): S = Q K^T and dP = dO V^T leave, per lane, 16
//               queries of one key; P and dS are the B operands of dV^T += dO^T P and dK^T += Q^T dS.
//               Q and dO tiles of 32 queries (with their lse and D) are staged in LDS.
// A staged tile is split once and read twice, by rows for the first products and by columns (transposing reads) for the second.
// The factor `scale` of dS is applied to the sums at the end.
//
// Bound: long sequences, the matrix pipe (seven products of 2 N^2 D per head for the five of the mathematics: S and dP are formed
// in both kernels): B2 H16 N2048 D128 busy in 70 % of the SIMD cycles, 4.2 vector instructions per matrix instruction.  At B8 H6 N789
// D64 33 % (dK/dV, one wave per SIMD) and 41 % (dQ): splitting, and few tiles per wave.
// Against the same kernels on v_mfma_f32_32x32x2_f32, whole backward, microseconds on one card: B2 H16 N2048 D128 2038 -> 1096,
// causal 1122 -> 594, D64 996 -> 570, causal D64 778 -> 332, B8 H6 N789 D64 347 -> 213, B8 H12 N197 D64 85 -> 51, B1 H12 N197 D64
// 34 -> 21, B1 H4 N4096 D128 causal 623 -> 487, with a mask B2 H12 N1024 D64 399 -> 195.  Relative error (2-norm, against float64)
// of dQ, dK, dV: N789 5.8, 5.7, 5.5e-7 -> 5.3, 5.2, 5.1e-7; B1 H16 N2048 D128 8.0, 8.0, 7.7e-7 -> 7.8, 7.8, 7.7e-7; of dQ at
// B2 H16 N2048 D128 1.08e-6 -> 9.2e-7.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "flash_f32.h"

namespace arhip {

struct FlashBwdParams {
    const float *q, *k, *v, *dout, *lse, *delta, *mask;
    const int32_t *kv_len;  // [B] or null
    float *dq, *dk, *dv;
    int Hq, Hkv, N;
    int nt;  // tiles per head: query tiles (dQ kernel) or key tiles (dK/dV kernel)
    int total_q, total_kv;  // workgroups in the dQ grid (nt * B * Hq) and in the dK/dV grid (nt * B * Hkv)
    int lpt_q, lpt_kv;  // causal: B * Hq / B * Hkv, and the grids run longest tile first over all heads; else 0
    int halves;  // 128 rows per workgroup: long sums are formed in two halves (bwd_first_half)
    float scale;
};

constexpr float BWD_LSE_FLOOR = -5e29f;  // lse at or below: the row saw no key (cuda_flash_train.rs:206)
constexpr float BWD_LOG2E = 1.44269504088896340736f;
// Gradients below 2^-80 are formed on the fp32 instruction: dS = P (dP - D) is split as well, and has lost no bit that counts in
// sums above that.
constexpr int BWD_TINY = -80;

// D[bh, i] = O[i] . dO[i], by D / 4 lanes of a wave, 16 bytes of the row each; their partial sums are added by a fixed
// butterfly.  Rows row0, row0 + 1, ... by lane group of the workgroup (D = 64: 16 rows, D = 128: 8; a wave per row, 4 bytes
// per lane, took 3.3 instead of 2.1 us on B8 H12 N197 D64).
template <int D>
constexpr int bwd_prep_rows() { return 256 / (D / 4); }
template <int D>
__device__ __forceinline__ void bwd_prep_row(const float *o, const float *dout, float *delta, long rows, long row, bool store)
{
    const int g = threadIdx.x & (D / 4 - 1);
    if (row >= rows) return;  // (whole lane groups)
    const float4 a = *(const float4 *)(o + row * D + 4 * g), b = *(const float4 *)(dout + row * D + 4 * g);
    float s = (a.x * b.x + a.y * b.y) + (a.z * b.z + a.w * b.w);
#pragma unroll
    for (int off = D / 8; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    if (store && g == 0) delta[row] = s;
}
// four rows per workgroup, the shape of the named entry's grid: the lane groups of a wave share a row
template <int D>
__device__ __forceinline__ void bwd_prep_body(const float *o, const float *dout, float *delta, long rows, long row0)
{
    bwd_prep_row<D>(o, dout, delta, rows, row0 + (threadIdx.x >> 6), (threadIdx.x & 63) < D / 4);
}

// One thread's share of a pair of 32-row tiles (A and B, e.g. K and V) between memory and LDS: items of 8 channels, the first
// half of them A's.  Rows past `last` repeat it (whatever they hold is multiplied by P = dS = 0).
template <int D, int T>
struct PairStage {
    using Tile = SplitTile<D>;
    static constexpr int ITEMS = 2 * Tile::ITEMS / T;  // per thread
    static constexpr int STEPS = (SPLIT_STEPS + 1) * ITEMS;  // of split_step
    static_assert(Tile::ITEMS % T == 0, "tile staging must divide evenly");
    float x[ITEMS][8];
    split8 sp;
    uint32_t tmp[4];

    static constexpr bool is_b(int j) { return j >= ITEMS / 2; }
    static __device__ __forceinline__ int item(int j, int t) { return t + (j - (is_b(j) ? ITEMS / 2 : 0)) * T; }
    __device__ __forceinline__ void fetch(const float *a, const float *b, int t, int row0, int last)
    {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const int it = item(j, t);
            const float *src = (is_b(j) ? b : a) + (size_t)min(row0 + Tile::item_row(it), last) * D + Tile::item_col(it);
            const float4 u = *(const float4 *)src, v = *(const float4 *)(src + 4);
            x[j][0] = u.x; x[j][1] = u.y; x[j][2] = u.z; x[j][3] = u.w;
            x[j][4] = v.x; x[j][5] = v.y; x[j][6] = v.z; x[j][7] = v.w;
        }
    }
    template <int I>
    __device__ __forceinline__ void split_step(unsigned char *ta, unsigned char *tb, int t)
    {
        constexpr int j = I / (SPLIT_STEPS + 1), k = I % (SPLIT_STEPS + 1);
        if constexpr (k < SPLIT_STEPS) split_op<k>(x[j], tmp, sp);
        else Tile::put(is_b(j) ? tb : ta, Tile::item_addr(item(j, t)), sp);
    }
    __device__ __forceinline__ void put(unsigned char *ta, unsigned char *tb, int t)
    {
        static_for<0, STEPS>([&](auto ic) __attribute__((always_inline)) { split_step<decltype(ic)::value>(ta, tb, t); });
    }
};

// LDS bytes of the bodies below.  Pipelined (128 queries / keys per workgroup): rings of tiles; SPLIT (32 per workgroup): a tile
// pair per wave, or the partial sums of the waves, which reuse it
template <int D, bool SPLIT>
constexpr int bwd_dq_lds_bytes()
{
    constexpr int merge = 4 * 32 * (D + 4) * 4, slabs = 4 * 2 * SplitTile<D>::BYTES;
    return (SPLIT ? (slabs > merge ? slabs : merge) : 5 * SplitTile<D>::BYTES) + 16;  // and a flag per wave
}
template <int D, bool SPLIT>
constexpr int bwd_dkv_lds_bytes()
{
    constexpr int merge = 4 * 2 * 32 * (D + 4) * 4, slabs = 4 * (2 * SplitTile<D>::BYTES + 256);
    return (SPLIT ? (slabs > merge ? slabs : merge) : 6 * SplitTile<D>::BYTES + 3 * 256) + 16;  // and a flag per wave
}

// 16 values per lane of a product of the first kind: c += A rows . B, A a tile in LDS
template <int D>
__device__ __forceinline__ f32x16 mul_rows(const unsigned char *tile, const int (&r_addr)[2], const split8 (&b)[D / 16])
{
    f32x16 c;
#pragma unroll
    for (int r = 0; r < 16; ++r) c[r] = 0.f;
#pragma unroll
    for (int st = 0; st < D / 16; ++st) c = mfma_split(SplitTile<D>::get_row(tile, r_addr[st & 1] + (st >> 1) * 2048), b[st], c);
    return c;
}
// acc += A columns . B
template <int D>
__device__ __forceinline__ void mul_cols(const unsigned char *tile, const int (&c_addr)[2], const split8 (&b)[2], f32x16 (&acc)[D / 32])
{
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
            const int o = db * 2048 + ks * 1024;
            acc[db] = mfma_split(SplitTile<D>::get_col(tile, c_addr[0] + o, c_addr[1] + o), b[ks], acc[db]);
        }
}

// A long sum is rounded with every matrix instruction, by an amount that grows with it.  So the sums over the first half of the
// tiles go to the place of the result they belong to, and are taken in again at the end, from 16 tiles on (causal, where most rows
// have shorter sums: from 48).  A third span, read back and added between two tiles, cost 5 to 12 % at head size 128, where it leaves
// values without a register.  row: the lane's row of the result.
template <bool CAUSAL>
__device__ __forceinline__ int bwd_first_half(int tiles, bool halves) { return halves && tiles >= (CAUSAL ? 48 : 16) ? tiles / 2 : 0; }
template <int D>
__device__ __forceinline__ void put_aside(float *row, int h, bool in_range, f32x16 (&acc)[D / 32])
{
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
            if (in_range)
                *(float4 *)(row + db * 32 + 8 * g + 4 * h) =
                    make_float4(acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
    }
}
template <int D>
__device__ __forceinline__ void take_in(const float *row, int h, f32x16 (&acc)[D / 32])
{
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float4 x = *(const float4 *)(row + db * 32 + 8 * g + 4 * h);
            acc[db][4 * g] += x.x; acc[db][4 * g + 1] += x.y; acc[db][4 * g + 2] += x.z; acc[db][4 * g + 3] += x.w;
        }
}

// dQ of 32 queries, and dK / dV of 32 keys, by one wave on v_mfma_f32_32x32x2_f32, which takes infinities and values at either
// end of the range as they are: for the workgroups whose operands are not the sum of three bf16 values (f32_split.h).  Operands
// straight from memory.
template <int D, bool CAUSAL>
__device__ __forceinline__ void bwd_dq_plain(const FlashBwdParams &p, const float *kp, const float *vp, int bh, int wq0, int kend)
{
    constexpr int DB = D / 32;
    const int lane = fresh_lane(), i32 = lane & 31, h = lane >> 5;
    const int N = p.N, q_row = wq0 + i32, rr = min(q_row, N - 1);
    if (wq0 >= N) return;
    const size_t qoff = ((size_t)bh * N + rr) * D + 4 * h;
    float4 q[D / 8], o[D / 8];
#pragma unroll
    for (int c = 0; c < D / 8; ++c) {
        q[c] = *(const float4 *)(p.q + qoff + 8 * c);
        o[c] = *(const float4 *)(p.dout + qoff + 8 * c);
    }
    const float lse = p.lse[(size_t)bh * N + rr], di = p.delta[(size_t)bh * N + rr];
    const bool live = lse > BWD_LSE_FLOOR;
    const float c2 = p.scale * BWD_LOG2E, lse2 = lse * BWD_LOG2E;
    f32x16_t acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
    const int all = (kend + F32_BK - 1) / F32_BK, tiles = CAUSAL ? min(all, wq0 / F32_BK + 1) : all;
#pragma clang loop unroll(disable)
    for (int it = 0; it < tiles; ++it) {
        const int k0 = it * F32_BK;
        const size_t off = (size_t)min(k0 + i32, kend - 1) * D + 4 * h;
        f32x16_t s, dp;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
        for (int c = 0; c < D / 8; ++c) {
            s = mfma_plain(*(const float4 *)(kp + off + 8 * c), q[c], s);
            dp = mfma_plain(*(const float4 *)(vp + off + 8 * c), o[c], dp);
        }
        // step r multiplies key 8 (r / 4) + 4 h + r % 4
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = k0 + 8 * (r >> 2) + 4 * h + (r & 3), kk = min(key, kend - 1);
            float x = fmaf(s[r], c2, -lse2);
            if (p.mask != nullptr) x = fmaf(p.mask[(size_t)rr * N + kk], BWD_LOG2E, x);
            const bool dead = key >= kend || (CAUSAL && key > q_row) || !live;
            const float ds = dead ? 0.f : __builtin_amdgcn_exp2f(x) * (dp[r] - di) * p.scale;
#pragma unroll
            for (int db = 0; db < DB; ++db)
                acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(key < kend ? kp[(size_t)kk * D + 32 * db + i32] : 0.f, ds, acc[db], 0, 0, 0);
        }
    }
    if (q_row >= N) return;
    float *op = p.dq + ((size_t)bh * N + q_row) * D;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *(float4 *)(op + db * 32 + 8 * g + 4 * h) = make_float4(acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]);
}

template <int D, bool CAUSAL>
__device__ __forceinline__ void bwd_dkv_plain(const FlashBwdParams &p, int b, int kvh, int wk0, int kvl)
{
    constexpr int DB = D / 32;
    const int lane = fresh_lane(), i32 = lane & 31, h = lane >> 5;
    const int N = p.N, key = wk0 + i32, jj = min(key, N - 1), group = p.Hq / p.Hkv;
    if (wk0 >= N) return;
    const size_t koff = (((size_t)b * p.Hkv + kvh) * N + jj) * D + 4 * h;
    float4 k[D / 8], v[D / 8];
#pragma unroll
    for (int c = 0; c < D / 8; ++c) {
        k[c] = *(const float4 *)(p.k + koff + 8 * c);
        v[c] = *(const float4 *)(p.v + koff + 8 * c);
    }
    const float c2 = p.scale * BWD_LOG2E;
    f32x16_t dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) dk[db][r] = dv[db][r] = 0.f;
    const int qt0 = CAUSAL ? wk0 / F32_BK : 0, per_head = (N + F32_BK - 1) / F32_BK - qt0;
    const int steps = wk0 < kvl ? group * per_head : 0;
#pragma clang loop unroll(disable)
    for (int st = 0; st < steps; ++st) {
        const size_t row0 = ((size_t)b * p.Hq + (size_t)kvh * group + st / per_head) * N;  // of the head
        const int q0 = (qt0 + st % per_head) * F32_BK;
        const size_t off = (row0 + min(q0 + i32, N - 1)) * D + 4 * h;
        f32x16_t s, dp;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
#pragma unroll
        for (int c = 0; c < D / 8; ++c) {
            s = mfma_plain(*(const float4 *)(p.q + off + 8 * c), k[c], s);
            dp = mfma_plain(*(const float4 *)(p.dout + off + 8 * c), v[c], dp);
        }
        // step r multiplies query 8 (r / 4) + 4 h + r % 4 of the tile
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int qi = q0 + 8 * (r >> 2) + 4 * h + (r & 3), qq = min(qi, N - 1);
            const float lse = p.lse[row0 + qq];
            float x = fmaf(s[r], c2, -lse * BWD_LOG2E);
            if (p.mask != nullptr) x = fmaf(p.mask[(size_t)qq * N + jj], BWD_LOG2E, x);
            const bool dead = qi >= N || key >= kvl || (CAUSAL && key > qi) || !(lse > BWD_LSE_FLOOR);
            const float pr = dead ? 0.f : __builtin_amdgcn_exp2f(x);
            const float ds = dead ? 0.f : pr * (dp[r] - p.delta[row0 + qq]) * p.scale;
            const size_t at = (row0 + qq) * D + i32;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                dv[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(qi < N ? p.dout[at + 32 * db] : 0.f, pr, dv[db], 0, 0, 0);
                dk[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(qi < N ? p.q[at + 32 * db] : 0.f, ds, dk[db], 0, 0, 0);
            }
        }
    }
    if (key >= N) return;
    const size_t out = (((size_t)b * p.Hkv + kvh) * N + key) * D;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d = db * 32 + 8 * g + 4 * h;
            *(float4 *)(p.dk + out + d) = make_float4(dk[db][4 * g], dk[db][4 * g + 1], dk[db][4 * g + 2], dk[db][4 * g + 3]);
            *(float4 *)(p.dv + out + d) = make_float4(dv[db][4 * g], dv[db][4 * g + 1], dv[db][4 * g + 2], dv[db][4 * g + 3]);
        }
}

// dQ.  lds: bwd_dq_lds_bytes<D, SPLIT>() bytes.  Workgroup wg_linear in [0, nt * B * Hq), four waves: 128 queries
// of one head.  SPLIT (few, short heads: one wave per workgroup would leave each SIMD a long chain of
// matrix instructions and most of the chip idle): the waves share the same 32 queries and deal the
// key tiles out between them (wave w takes tiles w, w + 4, ...), each staging its tiles in its own
// LDS slab with no workgroup barrier; the partial dQ of the waves are added through LDS in wave order.
// HAS_MASK: p.mask is not null.  The 16 mask values of a lane are requested where the logits they belong to are begun: asked for where
// they are added, their way from memory was waited for in every tile (whole backward, B1 H2 N1024 D128 253 -> 149 us, B2 H6
// N1500 D64 causal 300 -> 252, B2 H12 N1024 D64 318 -> 197).
template <int D, bool CAUSAL, bool SPLIT, bool HAS_MASK>
__device__ __forceinline__ void bwd_dq_body(const FlashBwdParams &p, unsigned char *lds, int wg_linear)
{
    constexpr int NW = 4;
    constexpr int BQ = SPLIT ? 32 : NW * 32;
    constexpr int DB = D / 32, KSTEPS = D / 16;
    using Tile = SplitTile<D>;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i32 = lane & 31, h = lane >> 5;
    // every XCD (consecutive workgroups go to different ones) gets a contiguous range of heads
    const int wg_x = (p.total_q > 0 && (p.total_q & 7) == 0) ? (wg_linear & 7) * (p.total_q >> 3) + (wg_linear >> 3) : wg_linear;
    int bh = wg_x / p.nt;
    int qt = wg_x - bh * p.nt;
    if (CAUSAL) qt = p.nt - 1 - qt;  // the longest query tiles first, within a head ...
    if (CAUSAL && p.lpt_q > 0) {     // ... or over the whole grid
        qt = p.nt - 1 - wg_linear / p.lpt_q;
        bh = wg_linear % p.lpt_q;
    }
    const int b = bh / p.Hq, head = bh - b * p.Hq;
    const int N = p.N;
    const int qblk = qt * BQ;
    const int wq0 = qblk + (SPLIT ? 0 : wave * 32);
    const int q_row = wq0 + i32;
    const int rr = min(q_row, N - 1);
    int kvl = N;
    if (p.kv_len) {
        kvl = p.kv_len[b];
        kvl = kvl < 0 ? 0 : (kvl > N ? N : kvl);
    }
    int kend = kvl;
    if (CAUSAL) kend = min(kend, min(N, qblk + BQ));
    const int ntiles = (kend + F32_BK - 1) / F32_BK;
    const int my_tiles = wq0 >= N ? 0 : CAUSAL ? min(ntiles, (wq0 + 31) / F32_BK + 1) : ntiles;
    const int kvh = head / (p.Hq / p.Hkv);
    const float *kp = p.k + ((size_t)b * p.Hkv + kvh) * (size_t)N * D;
    const float *vp = p.v + ((size_t)b * p.Hkv + kvh) * (size_t)N * D;
    const size_t qoff = ((size_t)bh * N + rr) * D + h * 8;

    // The first tiles are requested before the wave's own rows are waited for and split: one memory round trip, not two
    // (few or short heads: a round trip is a tenth of the kernel).
    PairStage<D, SPLIT ? 64 : NW * 64> first, stage;
    if constexpr (SPLIT) {
        if (wave < ntiles) stage.fetch(kp, vp, lane, wave * F32_BK, kend - 1);
    } else if (ntiles > 0) {
        first.fetch(kp, vp, tid, 0, kend - 1);
        stage.fetch(kp, vp, tid, F32_BK, kend - 1);
    }
    const float lse = p.lse[(size_t)bh * N + rr];
    const float di = p.delta[(size_t)bh * N + rr];
    ARHIP_FENCE();
    split8 qr[KSTEPS], dor[KSTEPS];
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
        qr[s] = split_8(*(const float4 *)(p.q + qoff + 16 * s), *(const float4 *)(p.q + qoff + 16 * s + 4));
        dor[s] = split_8(*(const float4 *)(p.dout + qoff + 16 * s), *(const float4 *)(p.dout + qoff + 16 * s + 4));
    }
    const bool beyond = beyond_split<KSTEPS>(qr) || beyond_split<KSTEPS>(dor);
    // P = exp(x - lse) as v_exp_f32 (base 2) of x * log2(e) - lse * log2(e), the second product unrounded (rounded, it would shift a
    // whole row of P by half a unit in its last place); a row that saw no key has P = 0
    const float c2 = p.scale * BWD_LOG2E, neg_lse = lse > BWD_LSE_FLOOR ? -lse : -__builtin_inff();

    f32x16_t acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.f;
    const int r_addr[2] = {Tile::row_addr(i32, h, 0), Tile::row_addr(i32, h, 1)};
    const int c_addr[2] = {Tile::col_addr(lane, 0), Tile::col_addr(lane, 1)};

    // S^T = K Q^T and dP^T = V dO^T: lane = query, register r = key 8 (r / 4) + 4 h + r % 4
    f32x16_t s, dp;
    float ds[16], t4[4];  // dS / scale; scratch of ds_step
    split8 db_[2];
    // what the logits are multiplied by in the exponent: c2, or 1 where the mask has been added (add_mask)
    const float cx = HAS_MASK ? 1.f : c2;
    float mv[16];
    const float *m_row = HAS_MASK ? p.mask + (size_t)rr * N : nullptr;
    auto fetch_mask = [&](int k0) __attribute__((always_inline)) {
        typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_u;  // rows of any N: 4-byte aligned
        if constexpr (!HAS_MASK) return;
        if (k0 + F32_BK <= N) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4_u v = *(const f32x4_u *)(m_row + k0 + 8 * g + 4 * h);
                mv[4 * g] = v[0]; mv[4 * g + 1] = v[1]; mv[4 * g + 2] = v[2]; mv[4 * g + 3] = v[3];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) mv[r] = m_row[min(k0 + 8 * (r >> 2) + 4 * h + (r & 3), N - 1)];
        }
        ARHIP_FENCE();
    };
    auto add_mask = [&]() __attribute__((always_inline)) {
        if constexpr (!HAS_MASK) return;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = fmaf(mv[r], BWD_LOG2E, s[r] * c2);
    };
    auto make_ds = [&](int r) __attribute__((always_inline)) {
        ds[r] = __builtin_amdgcn_exp2f(fmaf(neg_lse, BWD_LOG2E, s[r] * cx)) * (dp[r] - di);
    };
    // the same in steps 0 .. 23: exponents and exponentials two at a time, then the differences and the products four at a time
    auto ds_step = [&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value;
        if constexpr (i < 16) {
            constexpr int e = (i >> 1) * 2;
#pragma unroll
            for (int r = e; r < e + 2; ++r) ds[r] = (i & 1) ? __builtin_amdgcn_exp2f(ds[r]) : fmaf(neg_lse, BWD_LOG2E, s[r] * cx);
            pin(ds[e], ds[e + 1]);
        } else {
            constexpr int e = ((i - 16) >> 1) * 4;
#pragma unroll
            for (int r = e; r < e + 4; ++r) {
                float &v = (i & 1) ? ds[r] : t4[r - e];
                v = (i & 1) ? ds[r] * t4[r - e] : dp[r] - di;
                asm volatile("" : "+v"(v));
            }
        }
    };
    // keys past the end or above the diagonal have P = 0
    auto drop_dead = [&](int k0) __attribute__((always_inline)) {
        if (!(k0 + F32_BK > kend || (CAUSAL && k0 + F32_BK - 1 > wq0))) return;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int key = k0 + 8 * (r >> 2) + 4 * h + (r & 3);
            if (key >= kend || (CAUSAL && key > q_row)) ds[r] = 0.f;
        }
    };
    uint32_t tmp[4];
    auto split_ds = [&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, g = i / SPLIT_STEPS;
        split_op<i % SPLIT_STEPS>(ds + 8 * g, tmp, db_[g]);
    };

    if constexpr (SPLIT) {
        unsigned char *kt = lds + wave * 2 * Tile::BYTES, *vt = kt + Tile::BYTES;
        for (int it = wave; it < ntiles; it += NW) {
            const int k0 = it * F32_BK;
            stage.put(kt, vt, lane);
            fetch_mask(k0);
            if (it + NW < ntiles) stage.fetch(kp, vp, lane, k0 + NW * F32_BK, kend - 1);
            s = mul_rows<D>(kt, r_addr, qr);
            dp = mul_rows<D>(vt, r_addr, dor);
            add_mask();
#pragma unroll
            for (int r = 0; r < 16; ++r) make_ds(r);
            drop_dead(k0);
            static_for<0, 2 * SPLIT_STEPS>(split_ds);
            mul_cols<D>(kt, c_addr, db_, acc);
        }
    } else {
        // The pipelined tile loop (flash_f32.h), one tile ahead:
        //   R1(n)  S(n+1), dP(n+1)   (MFMA)  |  dS(n) split into its three parts; this thread's share of K(n+2), V(n+2) split
        //                                       and written to LDS                                  (VALU)
        //   R2(n)  dQ += K(n)^T dS(n) (MFMA)  |  dS(n+1) from S(n+1), dP(n+1)                        (VALU)
        // then a barrier.  K is read in two iterations (three tiles in LDS), V in one (two).
        unsigned char *k_ring = lds, *v_ring = lds + 3 * Tile::BYTES;
        if (ntiles > 0) {
            first.put(k_ring, v_ring, tid);
            stage.put(k_ring + Tile::BYTES, v_ring + Tile::BYTES, tid);
            stage.fetch(kp, vp, tid, 2 * F32_BK, kend - 1);
        }
        __syncthreads();
        if (my_tiles > 0) {
            fetch_mask(0);
            s = mul_rows<D>(k_ring, r_addr, qr);
            dp = mul_rows<D>(v_ring, r_addr, dor);
            add_mask();
#pragma unroll
            for (int r = 0; r < 16; ++r) make_ds(r);
            drop_dead(0);
        }
        __syncthreads();  // V(0) has been read: its slot is written next
        int k_cur = 0;  // ring slot of K(n)
        const int half = bwd_first_half<CAUSAL>(my_tiles, p.halves != 0);
        auto slot = [](int k) __attribute__((always_inline)) { return k >= 3 ? k - 3 : k; };
        SplitFrag fr;
        int n = 0;
        float *aside = p.dq + ((size_t)bh * N + rr) * D;
#pragma clang loop unroll(disable)
        for (int part = half > 0 ? 0 : 1; part < 2; ++part) {
            const int end = part == 0 ? half : my_tiles - 1;
#pragma clang loop unroll(disable)
            for (; n < end; ++n) {
                const unsigned char *kt = k_ring + k_cur * Tile::BYTES, *kt1 = k_ring + slot(k_cur + 1) * Tile::BYTES,
                                    *vt1 = v_ring + ((n + 1) & 1) * Tile::BYTES;
                unsigned char *kt2 = k_ring + slot(k_cur + 2) * Tile::BYTES, *vt2 = v_ring + (n & 1) * Tile::BYTES;
                auto load_row = [&](auto fi, auto pi, const unsigned char *tile, int st) __attribute__((always_inline)) {
                    constexpr int f = decltype(fi)::value, P = decltype(pi)::value;
                    fr.template set<(f & 1), P>(Tile::template get_row_part<P>(tile, r_addr[st & 1] + (st >> 1) * 2048));
                };
                auto load_col = [&](auto fi, auto pi, const unsigned char *tile, int i) __attribute__((always_inline)) {
                    constexpr int f = decltype(fi)::value, P = decltype(pi)::value;
                    const int o = (i % DB) * 2048 + (i / DB) * 1024;
                    fr.template set<(f & 1), P>(Tile::template get_col_part<P>(tile, c_addr[0] + o, c_addr[1] + o));
                };
                fetch_mask((n + 1) * F32_BK);
                // ---- R1 ----  (a few vector steps first: the first fragment has just become visible)
                static_for<0, 3>([&](auto pi) __attribute__((always_inline)) { load_row(std::integral_constant<int, 0>{}, pi, kt1, 0); });
                static_for<0, 4>(split_ds);
                ARHIP_FENCE();
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
                mfma_region<2 * KSTEPS, 2 * SPLIT_STEPS - 4 + PairStage<D, NW * 64>::STEPS>(
                    [&](auto fi, auto mi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value, m = decltype(mi)::value;
                        if constexpr (f < KSTEPS) s = mfma_split_step<m>(fr.template get<(f & 1)>(), qr[f], s);
                        else dp = mfma_split_step<m>(fr.template get<(f & 1)>(), dor[f - KSTEPS], dp);
                    },
                    [&](auto fi, auto pi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value;
                        if constexpr (f < KSTEPS) load_row(fi, pi, kt1, f);
                        else if constexpr (f < 2 * KSTEPS) load_row(fi, pi, vt1, f - KSTEPS);
                        else load_col(fi, pi, kt, 0);
                    },
                    [&](auto ic) __attribute__((always_inline)) {
                        constexpr int i = decltype(ic)::value;
                        if constexpr (i < 2 * SPLIT_STEPS - 4) split_ds(std::integral_constant<int, i + 4>{});
                        else stage.template split_step<i - (2 * SPLIT_STEPS - 4)>(kt2, vt2, tid);
                    });
                if (n + 3 < ntiles) stage.fetch(kp, vp, tid, (n + 3) * F32_BK, kend - 1);
                add_mask();
                // ---- R2 ----
                mfma_region<2 * DB, 24>(
                    [&](auto fi, auto mi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value;
                        acc[f % DB] = mfma_split_step<decltype(mi)::value>(fr.template get<(f & 1)>(), db_[f / DB], acc[f % DB]);
                    },
                    [&](auto fi, auto pi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value;
                        if constexpr (f < 2 * DB) load_col(fi, pi, kt, f);
                    },
                    ds_step);
                drop_dead((n + 1) * F32_BK);
                k_cur = slot(k_cur + 1);
                __syncthreads();
            }
            if (part == 0) put_aside<D>(aside, h, q_row < N, acc);
        }
        if (my_tiles > 0) {
            static_for<0, 2 * SPLIT_STEPS>(split_ds);
            mul_cols<D>(k_ring + k_cur * Tile::BYTES, c_addr, db_, acc);
            if (half > 0) take_in<D>(aside, h, acc);
        }
        // under the causal mask a wave is done before others of its workgroup: it still stages tiles for them
        for (; n < ntiles - 1; ++n) {
            stage.put(k_ring + slot(k_cur + 2) * Tile::BYTES, v_ring + (n & 1) * Tile::BYTES, tid);
            if (n + 3 < ntiles) stage.fetch(kp, vp, tid, (n + 3) * F32_BK, kend - 1);
            k_cur = slot(k_cur + 1);
            __syncthreads();
        }
    }

    uint32_t *flags = (uint32_t *)(lds + bwd_dq_lds_bytes<D, SPLIT>() - 16);
    ResultRange results;
    if constexpr (SPLIT) {
        // the waves' partial sums, each as [32 queries][ROW]
        constexpr int ROW = D + 4, SLAB = 32 * ROW;
        float *part = (float *)lds;
        __syncthreads();  // every wave's tiles are consumed
        float *ow = part + wave * SLAB;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(float4 *)&ow[i32 * ROW + db * 32 + 8 * g + 4 * h] =
                    make_float4(acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]);
        __syncthreads();
        // thread t: query t % 32, channels [cg * CPT, cg * CPT + CPT)
        constexpr int CPT = D / (NW * 2);
        static_assert(CPT % 4 == 0, "whole float4s per thread");
        const int q = tid & 31, cg = tid >> 5;
        float4 sum[CPT / 4];
#pragma unroll
        for (int c = 0; c < CPT / 4; ++c) {
            sum[c] = *(const float4 *)&part[q * ROW + cg * CPT + 4 * c];
#pragma unroll
            for (int w = 1; w < NW; ++w) {
                const float4 x = *(const float4 *)&part[w * SLAB + q * ROW + cg * CPT + 4 * c];
                sum[c].x += x.x; sum[c].y += x.y; sum[c].z += x.z; sum[c].w += x.w;
            }
            results.take(sum[c]);
        }
        // operands that are not the sum of three bf16 values
        flag_write(flags, wave, results.beyond<BWD_TINY>() || beyond);
        __syncthreads();
        if (__builtin_expect(flag_read<NW>(flags), 0)) {
            if (wave == 0) bwd_dq_plain<D, CAUSAL>(p, kp, vp, bh, fresh(wq0), kend);
            return;
        }
        if (qblk + q < N) {
            float *op = p.dq + ((size_t)bh * N + qblk + q) * D + cg * CPT;
#pragma unroll
            for (int c = 0; c < CPT / 4; ++c)
                *(float4 *)(op + 4 * c) = make_float4(sum[c].x * p.scale, sum[c].y * p.scale, sum[c].z * p.scale, sum[c].w * p.scale);
        }
        return;
    }
    if (q_row < N) {
        float *op = p.dq + ((size_t)bh * N + q_row) * D;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(float4 *)(op + db * 32 + 8 * g + 4 * h) = make_float4(acc[db][4 * g] * p.scale, acc[db][4 * g + 1] * p.scale,
                                                                        acc[db][4 * g + 2] * p.scale, acc[db][4 * g + 3] * p.scale);
    }
    // operands that are not the sum of three bf16 values: the results are formed again, by the lanes that stored them
#pragma unroll
    for (int db = 0; db < DB; ++db) results.take(acc[db]);
    flag_write(flags, wave, results.beyond<BWD_TINY>() || beyond);
    __syncthreads();
    if (__builtin_expect(flag_read<NW>(flags), 0)) {
        wait_vmem_le<0>();
        bwd_dq_plain<D, CAUSAL>(p, kp, vp, bh, fresh(wq0), kend);
    }
}

// dK and dV.  Workgroup wg_linear in [0, nt * B * Hkv), four waves: 128 keys of one K/V head.  SPLIT: the waves
// share the same 32 keys and deal the (head of the group, query tile) steps out between them, each in
// its own LDS slab; the partial dK and dV of the waves are added through LDS in wave order.
template <int D, bool CAUSAL, bool SPLIT, bool HAS_MASK>
__device__ __forceinline__ void bwd_dkv_body(const FlashBwdParams &p, unsigned char *lds, int wg_linear)
{
    constexpr int NW = 4;
    constexpr int BKW = SPLIT ? 32 : NW * 32;  // keys per workgroup
    constexpr int DB = D / 32, KSTEPS = D / 16;
    using Tile = SplitTile<D>;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int stid = SPLIT ? lane : tid;      // index among the threads staging a tile
    const int i32 = lane & 31, h = lane >> 5;
    const int wg_x = (p.total_kv > 0 && (p.total_kv & 7) == 0) ? (wg_linear & 7) * (p.total_kv >> 3) + (wg_linear >> 3) : wg_linear;
    int kv_bh = wg_x / p.nt;
    int kt = wg_x - kv_bh * p.nt;  // causal: the first key tiles see the most queries
    if (CAUSAL && p.lpt_kv > 0) {       // the longest over the whole grid first
        kt = wg_linear / p.lpt_kv;
        kv_bh = wg_linear % p.lpt_kv;
    }
    const int b = kv_bh / p.Hkv, kvh = kv_bh - b * p.Hkv;
    const int group = p.Hq / p.Hkv;
    const int N = p.N;
    const int kblk = kt * BKW;
    const int wk0 = kblk + (SPLIT ? 0 : wave * 32);
    const int key = wk0 + i32;
    const int jj = min(key, N - 1);
    int kvl = N;
    if (p.kv_len) {
        kvl = p.kv_len[b];
        kvl = kvl < 0 ? 0 : (kvl > N ? N : kvl);
    }
    const bool key_live = key < kvl;
    const float c2 = p.scale * BWD_LOG2E;

    f32x16_t dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) dk[db][r] = dv[db][r] = 0.f;
    const int r_addr[2] = {Tile::row_addr(i32, h, 0), Tile::row_addr(i32, h, 1)};
    const int c_addr[2] = {Tile::col_addr(lane, 0), Tile::col_addr(lane, 1)};

    // queries before the workgroup's first key see none of its keys under the causal mask
    const int qt0 = CAUSAL ? kblk / F32_BK : 0;
    const int qtiles = (N + F32_BK - 1) / F32_BK, per_head = qtiles - qt0;
    // (head of the group, query tile) pairs, head-major; a workgroup whose keys are all past the key length has none
    const int steps = kblk < kvl ? group * per_head : 0;
    // the last query tile first, so that under the causal mask the tiles a wave has no part in come at the end of a head
    auto step_head = [&](int st) __attribute__((always_inline)) { return (size_t)b * p.Hq + (size_t)kvh * group + st / per_head; };
    auto step_q0 = [&](int st) __attribute__((always_inline)) { return (qtiles - 1 - st % per_head) * F32_BK; };

    PairStage<D, SPLIT ? 64 : NW * 64> first, stage;
    float st_l[2] = {0.f, 0.f}, st_d[2] = {0.f, 0.f};
    auto fetch_tiles = [&](decltype(stage) &to, int st) __attribute__((always_inline)) {
        const size_t off = step_head(st) * N * D;
        to.fetch(p.q + off, p.dout + off, stid, step_q0(st), N - 1);
    };
    // -lse; rows that saw no key (and rows past the end) have P = 0
    auto fetch_stats = [&](int st, int to = 0) __attribute__((always_inline)) {
        if (stid < F32_BK) {
            const size_t at = step_head(st) * N + min(step_q0(st) + stid, N - 1);
            st_l[to] = p.lse[at];
            st_d[to] = p.delta[at];
        }
    };
    auto put_stats = [&](float *stat, int st, int from = 0) __attribute__((always_inline)) {
        if (stid < F32_BK) {
            const bool live = step_q0(st) + stid < N;
            stat[stid] = live && st_l[from] > BWD_LSE_FLOOR ? -st_l[from] : -__builtin_inff();
            stat[32 + stid] = live ? st_d[from] : 0.f;
        }
    };
    // The first tiles are requested before the wave's own rows are waited for and split: one memory round trip, not three.
    if constexpr (SPLIT) {
        if (wave < steps) {
            fetch_tiles(stage, wave);
            fetch_stats(wave);
        }
    } else if (steps > 0) {
        fetch_tiles(first, 0);
        fetch_stats(0, 0);
        fetch_tiles(stage, min(1, steps - 1));
        fetch_stats(min(1, steps - 1), 1);
    }
    ARHIP_FENCE();
    split8 kr[KSTEPS], vr[KSTEPS];
    {
        const size_t off = ((size_t)kv_bh * N + jj) * D + h * 8;
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
            kr[s] = split_8(*(const float4 *)(p.k + off + 16 * s), *(const float4 *)(p.k + off + 16 * s + 4));
            vr[s] = split_8(*(const float4 *)(p.v + off + 16 * s), *(const float4 *)(p.v + off + 16 * s + 4));
        }
    }
    const bool beyond = beyond_split<KSTEPS>(kr) || beyond_split<KSTEPS>(vr);

    // S = Q K^T and dP = dO V^T: lane = key, register r = query 8 (r / 4) + 4 h + r % 4 of the tile
    f32x16_t s, dp;
    float pr[16], ds[16];  // P and dS / scale
    float4 st4[4];         // lse, then D, of the lane's 16 queries
    split8 pb[2], db_[2];
    auto read_stats = [&](const float *stat) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < 4; ++g) st4[g] = *(const float4 *)&stat[8 * g + 4 * h];
    };
    auto stat_of = [&](int r) __attribute__((always_inline)) {
        const float4 &v = st4[r >> 2];
        return (r & 3) == 0 ? v.x : (r & 3) == 1 ? v.y : (r & 3) == 2 ? v.z : v.w;
    };
    // what the logits are multiplied by in the exponent: c2, or 1 where the mask has been added (add_mask)
    const float cx = HAS_MASK ? 1.f : c2;
    float mv[16];
    auto fetch_mask = [&](int q0) __attribute__((always_inline)) {
        if constexpr (!HAS_MASK) return;
#pragma unroll
        for (int r = 0; r < 16; ++r) mv[r] = p.mask[(size_t)min(q0 + 8 * (r >> 2) + 4 * h + (r & 3), N - 1) * N + jj];
        ARHIP_FENCE();
    };
    auto add_mask = [&]() __attribute__((always_inline)) {
        if constexpr (!HAS_MASK) return;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = fmaf(mv[r], BWD_LOG2E, s[r] * c2);
    };
    auto make_p = [&](int r) __attribute__((always_inline)) { pr[r] = __builtin_amdgcn_exp2f(fmaf(stat_of(r), BWD_LOG2E, s[r] * cx)); };
    auto make_ds = [&](int r) __attribute__((always_inline)) { ds[r] = pr[r] * (dp[r] - stat_of(r)); };
    // keys past the key length or below the diagonal have P = 0
    auto drop_dead = [&](int q0) __attribute__((always_inline)) {
        if (!(wk0 + 31 >= kvl || (CAUSAL && wk0 + 31 > q0))) return;
        const int kq = key - q0 - 4 * h;  // causal: query 8 gq + 4 h + t of the tile sees this lane's key iff kq <= 8 gq + t
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (!key_live || (CAUSAL && kq > 8 * (r >> 2) + (r & 3))) pr[r] = ds[r] = 0.f;
    };
    auto make_all = [&](int q0, const float *stat) __attribute__((always_inline)) {
        add_mask();
        read_stats(stat);
#pragma unroll
        for (int r = 0; r < 16; ++r) make_p(r);
        read_stats(stat + 32);
#pragma unroll
        for (int r = 0; r < 16; ++r) make_ds(r);
        drop_dead(q0);
    };
    uint32_t tmp[4];
    auto split_p = [&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, g = i / SPLIT_STEPS;
        split_op<i % SPLIT_STEPS>(pr + 8 * g, tmp, pb[g]);
    };
    auto split_ds = [&](auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, g = i / SPLIT_STEPS;
        split_op<i % SPLIT_STEPS>(ds + 8 * g, tmp, db_[g]);
    };

    if constexpr (SPLIT) {
        unsigned char *qs = lds + wave * (2 * Tile::BYTES + 256), *dos = qs + Tile::BYTES;
        float *stat = (float *)(qs + 2 * Tile::BYTES);
        for (int st = wave; st < steps; st += NW) {
            stage.put(qs, dos, lane);
            put_stats(stat, st);
            if (st + NW < steps) {
                fetch_tiles(stage, st + NW);
                fetch_stats(st + NW);
            }
            fetch_mask(step_q0(st));
            s = mul_rows<D>(qs, r_addr, kr);
            dp = mul_rows<D>(dos, r_addr, vr);
            make_all(step_q0(st), stat);
            static_for<0, 2 * SPLIT_STEPS>(split_p);
            mul_cols<D>(dos, c_addr, pb, dv);
            static_for<0, 2 * SPLIT_STEPS>(split_ds);
            mul_cols<D>(qs, c_addr, db_, dk);
        }
    } else {
        // The pipelined loop (flash_f32.h), one step ahead:
        //   R1(n)  S(n+1), dP(n+1)                            (MFMA)  |  P(n) and dS(n) split into their three parts   (VALU)
        //   R2(n)  dV += dO(n)^T P(n), dK += Q(n)^T dS(n)      (MFMA)  |  P(n+1), dS(n+1); this thread's share of Q(n+2), dO(n+2)
        //                                                                split and written to LDS                     (VALU)
        // then a barrier.  Both tiles are read in two iterations: rings of three.
        unsigned char *q_ring = lds, *o_ring = lds + 3 * Tile::BYTES;
        float *stats = (float *)(lds + 6 * Tile::BYTES);
        // steps this wave computes on (heads sharing the K/V head: all but those at the very end)
        const int mine = wk0 >= kvl ? 0 : CAUSAL ? max(0, steps - wave) : steps;
        if (steps > 0) {
            first.put(q_ring, o_ring, tid);
            put_stats(stats, 0, 0);
            if (steps > 1) {
                stage.put(q_ring + Tile::BYTES, o_ring + Tile::BYTES, tid);
                put_stats(stats + 64, 1, 1);
            }
            if (steps > 2) {
                fetch_tiles(stage, 2);
                fetch_stats(2);
            }
        }
        __syncthreads();
        if (mine > 0) {
            fetch_mask(step_q0(0));
            s = mul_rows<D>(q_ring, r_addr, kr);
            dp = mul_rows<D>(o_ring, r_addr, vr);
            make_all(step_q0(0), stats);
        }
        int cur = 0;  // ring slot of step n
        const int half = bwd_first_half<CAUSAL>(mine, p.halves != 0);
        float *k_aside = p.dk + ((size_t)kv_bh * N + jj) * D, *v_aside = p.dv + ((size_t)kv_bh * N + jj) * D;
        auto slot = [](int k) __attribute__((always_inline)) { return k >= 3 ? k - 3 : k; };
        SplitFrag fr;
        int n = 0;
#pragma clang loop unroll(disable)
        for (int part = half > 0 ? 0 : 1; part < 2; ++part) {
            const int end = part == 0 ? half : mine - 1;
#pragma clang loop unroll(disable)
            for (; n < end; ++n) {
                const int s1 = slot(cur + 1), s2 = slot(cur + 2);
                const unsigned char *qt = q_ring + cur * Tile::BYTES, *ot = o_ring + cur * Tile::BYTES;
                const unsigned char *qt1 = q_ring + s1 * Tile::BYTES, *ot1 = o_ring + s1 * Tile::BYTES;
                unsigned char *qt2 = q_ring + s2 * Tile::BYTES, *ot2 = o_ring + s2 * Tile::BYTES;
                auto load_row = [&](auto fi, auto pi, const unsigned char *tile, int st) __attribute__((always_inline)) {
                    constexpr int f = decltype(fi)::value, P = decltype(pi)::value;
                    fr.template set<(f & 1), P>(Tile::template get_row_part<P>(tile, r_addr[st & 1] + (st >> 1) * 2048));
                };
                auto load_col = [&](auto fi, auto pi, const unsigned char *tile, int i) __attribute__((always_inline)) {
                    constexpr int f = decltype(fi)::value, P = decltype(pi)::value;
                    const int o = (i % DB) * 2048 + (i / DB) * 1024;
                    fr.template set<(f & 1), P>(Tile::template get_col_part<P>(tile, c_addr[0] + o, c_addr[1] + o));
                };
                fetch_mask(step_q0(n + 1));
                // ---- R1 ----  (a few vector steps first: the first fragment has just become visible)
                static_for<0, 3>([&](auto pi) __attribute__((always_inline)) { load_row(std::integral_constant<int, 0>{}, pi, qt1, 0); });
                static_for<0, 4>(split_p);
                ARHIP_FENCE();
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
                mfma_region<2 * KSTEPS, 4 * SPLIT_STEPS - 4>(
                    [&](auto fi, auto mi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value, m = decltype(mi)::value;
                        if constexpr (f < KSTEPS) s = mfma_split_step<m>(fr.template get<(f & 1)>(), kr[f], s);
                        else dp = mfma_split_step<m>(fr.template get<(f & 1)>(), vr[f - KSTEPS], dp);
                    },
                    [&](auto fi, auto pi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value;
                        if constexpr (f < KSTEPS) load_row(fi, pi, qt1, f);
                        else if constexpr (f < 2 * KSTEPS) load_row(fi, pi, ot1, f - KSTEPS);
                        else load_col(fi, pi, ot, 0);
                    },
                    [&](auto ic) __attribute__((always_inline)) {
                        constexpr int i = decltype(ic)::value;
                        if constexpr (i < 2 * SPLIT_STEPS - 4) split_p(std::integral_constant<int, i + 4>{});
                        else split_ds(std::integral_constant<int, i - (2 * SPLIT_STEPS - 4)>{});
                    });
                add_mask();
                read_stats(stats + s1 * 64);
                // ---- R2 ----
                constexpr int CONV = decltype(stage)::STEPS;
                mfma_region<4 * DB, 24 + CONV>(
                    [&](auto fi, auto mi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value, m = decltype(mi)::value, g = f % (2 * DB);
                        if constexpr (f < 2 * DB) dv[g % DB] = mfma_split_step<m>(fr.template get<(f & 1)>(), pb[g / DB], dv[g % DB]);
                        else dk[g % DB] = mfma_split_step<m>(fr.template get<(f & 1)>(), db_[g / DB], dk[g % DB]);
                    },
                    [&](auto fi, auto pi) __attribute__((always_inline)) {
                        constexpr int f = decltype(fi)::value;
                        if constexpr (f < 2 * DB) load_col(fi, pi, ot, f);
                        else if constexpr (f < 4 * DB) load_col(fi, pi, qt, f - 2 * DB);
                    },
                    [&](auto ic) __attribute__((always_inline)) {
                        constexpr int i = decltype(ic)::value;
                        if constexpr (i < 16) {
                            constexpr int e = (i >> 1) * 2;
#pragma unroll
                            for (int r = e; r < e + 2; ++r) pr[r] = (i & 1) ? __builtin_amdgcn_exp2f(pr[r]) : fmaf(stat_of(r), BWD_LOG2E, s[r] * cx);
                            pin(pr[e], pr[e + 1]);
                            if constexpr (i == 15) read_stats(stats + s1 * 64 + 32);
                        } else if constexpr (i < 24) {
                            constexpr int e = ((i - 16) >> 1) * 4;
#pragma unroll
                            for (int r = e; r < e + 4; ++r) {
                                ds[r] = (i & 1) ? pr[r] * ds[r] : dp[r] - stat_of(r);
                                asm volatile("" : "+v"(ds[r]));
                            }
                        } else {
                            stage.template split_step<i - 24>(qt2, ot2, tid);
                        }
                    });
                if (n + 2 < steps) put_stats(stats + s2 * 64, n + 2);
                if (n + 3 < steps) {
                    fetch_tiles(stage, n + 3);
                    fetch_stats(n + 3);
                }
                drop_dead(step_q0(n + 1));
                cur = s1;
                __syncthreads();
            }
            if (part == 0) {
                put_aside<D>(k_aside, h, key < N, dk);
                put_aside<D>(v_aside, h, key < N, dv);
            }
        }
        if (mine > 0) {
            static_for<0, 2 * SPLIT_STEPS>(split_p);
            mul_cols<D>(o_ring + cur * Tile::BYTES, c_addr, pb, dv);
            static_for<0, 2 * SPLIT_STEPS>(split_ds);
            mul_cols<D>(q_ring + cur * Tile::BYTES, c_addr, db_, dk);
            if (half > 0) {
                take_in<D>(k_aside, h, dk);
                take_in<D>(v_aside, h, dv);
            }
        }
        // a wave that is done before others of its workgroup still stages tiles for them
        for (; n < steps - 1; ++n) {
            const int s2 = slot(cur + 2);
            if (n + 2 < steps) {
                stage.put(q_ring + s2 * Tile::BYTES, o_ring + s2 * Tile::BYTES, tid);
                put_stats(stats + s2 * 64, n + 2);
            }
            if (n + 3 < steps) {
                fetch_tiles(stage, n + 3);
                fetch_stats(n + 3);
            }
            cur = slot(cur + 1);
            __syncthreads();
        }
    }

    uint32_t *flags = (uint32_t *)(lds + bwd_dkv_lds_bytes<D, SPLIT>() - 16);
    ResultRange results;
    if constexpr (SPLIT) {
        // the waves' partial sums: dK, then dV, each as [32 keys][ROW]
        constexpr int ROW = D + 4, SLAB = 2 * 32 * ROW;
        float *part = (float *)lds;
        __syncthreads();  // every wave's tiles are consumed
        float *ow = part + wave * SLAB;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d = db * 32 + 8 * g + 4 * h;
                *(float4 *)&ow[i32 * ROW + d] = make_float4(dk[db][4 * g], dk[db][4 * g + 1], dk[db][4 * g + 2], dk[db][4 * g + 3]);
                *(float4 *)&ow[(32 + i32) * ROW + d] = make_float4(dv[db][4 * g], dv[db][4 * g + 1], dv[db][4 * g + 2], dv[db][4 * g + 3]);
            }
        __syncthreads();
        // thread t: key t % 32, channels [cg * CPT, cg * CPT + CPT) of dK and of dV
        constexpr int CPT = D / (NW * 2);
        static_assert(CPT % 4 == 0, "whole float4s per thread");
        const int kq = tid & 31, cg = tid >> 5;
        float4 sum[2][CPT / 4];
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int c = 0; c < CPT / 4; ++c) {
                float4 &y = sum[half][c];
                y = *(const float4 *)&part[(half * 32 + kq) * ROW + cg * CPT + 4 * c];
#pragma unroll
                for (int w = 1; w < NW; ++w) {
                    const float4 x = *(const float4 *)&part[w * SLAB + (half * 32 + kq) * ROW + cg * CPT + 4 * c];
                    y.x += x.x; y.y += x.y; y.z += x.z; y.w += x.w;
                }
                results.take(y);
            }
        // operands that are not the sum of three bf16 values
        flag_write(flags, wave, results.beyond<BWD_TINY>() || beyond);
        __syncthreads();
        if (__builtin_expect(flag_read<NW>(flags), 0)) {
            if (wave == 0) bwd_dkv_plain<D, CAUSAL>(p, b, kvh, fresh(wk0), kvl);
            return;
        }
        if (kblk + kq < N) {
            const size_t orow = ((size_t)kv_bh * N + kblk + kq) * D + cg * CPT;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                float *op = (half ? p.dv : p.dk) + orow;
                const float f = half ? 1.f : p.scale;
#pragma unroll
                for (int c = 0; c < CPT / 4; ++c) {
                    const float4 &y = sum[half][c];
                    *(float4 *)(op + 4 * c) = make_float4(y.x * f, y.y * f, y.z * f, y.w * f);
                }
            }
        }
        return;
    }
    if (key < N) {
        float *okp = p.dk + ((size_t)kv_bh * N + key) * D;
        float *ovp = p.dv + ((size_t)kv_bh * N + key) * D;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d = db * 32 + 8 * g + 4 * h;
                *(float4 *)(okp + d) = make_float4(dk[db][4 * g] * p.scale, dk[db][4 * g + 1] * p.scale, dk[db][4 * g + 2] * p.scale,
                                                   dk[db][4 * g + 3] * p.scale);
                *(float4 *)(ovp + d) = make_float4(dv[db][4 * g], dv[db][4 * g + 1], dv[db][4 * g + 2], dv[db][4 * g + 3]);
            }
    }
    // operands that are not the sum of three bf16 values: the results are formed again, by the lanes that stored them
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        results.take(dk[db]);
        results.take(dv[db]);
    }
    flag_write(flags, wave, results.beyond<BWD_TINY>() || beyond);
    __syncthreads();
    if (__builtin_expect(flag_read<NW>(flags), 0)) {
        wait_vmem_le<0>();
        bwd_dkv_plain<D, CAUSAL>(p, b, kvh, fresh(wk0), kvl);
    }
}

template <int D>
__global__ void __launch_bounds__(256) bwd_prep_kernel(const float *o, const float *dout, float *delta, long rows)
{
    bwd_prep_row<D>(o, dout, delta, rows, (long)blockIdx.x * bwd_prep_rows<D>() + threadIdx.x / (D / 4), true);
}

// dK/dV and dQ in one grid: workgroups [0, total_kv) form dK/dV, which takes longer, the others dQ.  They have nothing to
// do with each other, so where either grid alone leaves compute units idle (few or short heads, the end of any grid) the other's
// workgroups run there; and it is a launch fewer.  Forward and backward, us: B1 H12 N197 D64 26 -> 24, B2 H16 N2048 D128 causal
// 817 -> 800.
template <int D, bool CAUSAL, bool SPLIT, bool HAS_MASK>
__global__ void __launch_bounds__(256, 1) bwd_kernel(const FlashBwdParams p)
{
    constexpr int LQ = bwd_dq_lds_bytes<D, SPLIT>(), LKV = bwd_dkv_lds_bytes<D, SPLIT>();
    __shared__ __attribute__((aligned(16))) unsigned char lds[LQ > LKV ? LQ : LKV];
    const int wg = (int)blockIdx.x;
    if (wg < p.total_kv) bwd_dkv_body<D, CAUSAL, SPLIT, HAS_MASK>(p, lds, wg);
    else bwd_dq_body<D, CAUSAL, SPLIT, HAS_MASK>(p, lds, wg - p.total_kv);
}

// Head size 64, 128 rows per workgroup: dQ fits 256 registers, so that a SIMD holds two of its waves, and dK/dV does not.  In one
// kernel either dQ would lose its second wave or dK/dV spill 73 registers (B8 H12 N197: 41 us together, 16 + 23 one after the other).
template <bool CAUSAL, bool HAS_MASK>
__global__ void __launch_bounds__(256, 2) bwd_dq_kernel(const FlashBwdParams p)
{
    __shared__ __attribute__((aligned(16))) unsigned char lds[bwd_dq_lds_bytes<64, false>()];
    bwd_dq_body<64, CAUSAL, false, HAS_MASK>(p, lds, (int)blockIdx.x);
}

template <bool CAUSAL, bool HAS_MASK>
__global__ void __launch_bounds__(256, 1) bwd_dkv_kernel(const FlashBwdParams p)
{
    __shared__ __attribute__((aligned(16))) unsigned char lds[bwd_dkv_lds_bytes<64, false>()];
    bwd_dkv_body<64, CAUSAL, false, HAS_MASK>(p, lds, (int)blockIdx.x);
}

// The kernels of a backward pass behind the row scalar
template <bool HAS_MASK>
void launch_bwd(hipStream_t stream, const FlashBwdParams &p, int D, bool causal, bool split)
{
    auto go = [&](auto d, auto c) {
        constexpr int DD = decltype(d)::value;
        constexpr bool C = decltype(c)::value;
        const dim3 block(256), q_grid((unsigned)p.total_q), kv_grid((unsigned)p.total_kv), both((unsigned)(p.total_kv + p.total_q));
        if (DD == 128 || split) {
            hipLaunchKernelGGL((bwd_kernel<DD, C, DD == 64, HAS_MASK>), both, block, 0, stream, p);
        } else {
            hipLaunchKernelGGL((bwd_dq_kernel<C, HAS_MASK>), q_grid, block, 0, stream, p);
            hipLaunchKernelGGL((bwd_dkv_kernel<C, HAS_MASK>), kv_grid, block, 0, stream, p);
        }
    };
    auto by_mask = [&](auto d) { causal ? go(d, std::true_type{}) : go(d, std::false_type{}); };
    D == 64 ? by_mask(std::integral_constant<int, 64>{}) : by_mask(std::integral_constant<int, 128>{});
}

}  // namespace arhip
