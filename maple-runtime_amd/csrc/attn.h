// attn.h -- the attention half of a Maple layer on the card (gfull_attn): per-head norms, rope and the fp16
// key/value cache, then causal grouped-query attention, for one sequence whose chunk of nb tokens sits at
// positions pos0 .. pos0+nb-1. The arithmetic follows maple.c's step_batch (maple.c:706-724) in the order
// the oracle's mo_attn_chunk fixes (oracle/moe_oracle.c), so the results equal the oracle's bit for bit:
//   head rmsnorm  maple.c:398-402 with n = 128: fp64 sum of squares in index order
//   rope          maple.c:403-411, in the FMA-contracted form maple.c's build computes
//   fp16 cache    maple.c:314-320, round to nearest even (v kept widened to fp32)
//   attention     maple.c:516-558 (attend_group, AVX2 path): scores as 8 FMA lanes over the head dimension
//                 folded by hsum8, softmax with the library's exp and a sum in position order, output as an
//                 FMA chain over positions.
// Work split: scores and the weighted sum of values run on the f32 matrix cores in tiles of 16 rows, 4 consecutive tokens
// x the 4 query heads of one key/value head, so each cached key or value row is read once for the tile; a
// token's own window is enforced with a zero weight outside it (an FMA with weight 0 and a finite value leaves a chain
// unchanged, exactly), so a tile shares one loop over positions. Values past fp16's range are infinities in the cache: a
// tile with such a position at the ends of its windows takes its tokens one by one (att_pv_tokens).
#pragma once
#include <hip/hip_fp16.h>
#include "kernels.h"

#define AT_HD 128
#define AT_QKV 3072   // q 16 x 128 | k 4 x 128 | v 4 x 128 per token
#define AT_XS 129     // LDS row stride of a head (a lane per head reads its own row without bank conflicts)

__device__ __forceinline__ int att_lo(int pos, int glob, int win) { return glob ? 0 : (pos - win > 0 ? pos - win : 0); }

// Raises *a to v (float maximum through integer atomics: non-negative floats order as signed integers,
// negative ones in reverse as unsigned integers).
__device__ __forceinline__ void atomic_max_f32(float *a, float v) {
    if (__float_as_int(v) >= 0) atomicMax((int *)a, __float_as_int(v));
    else atomicMin((unsigned int *)a, __float_as_uint(v));
}

// The key cache of one head (fp16), in blocks of 16 positions (2048 values) laid out as k_att_scores' MFMAs load them: dim
// d = (4 s + g) * 8 + j of the block's position att_perm(m) at ((s * 4 + g) * 16 + m) * 8 + j, so lane (g, m)'s 4 loads of 16
// bytes are 1 KB runs over the wave. (In rows of positions each group of 4 lanes reads 4 rows: four times the L1 lookups.)
#define AT_KBLK (16 * AT_HD)
__device__ __forceinline__ int att_perm(int m) { return 4 * (m & 3) + (m >> 2); }   // its own inverse
__device__ __forceinline__ int att_kidx(int pos, int d) {
    return (pos >> 4) * AT_KBLK + ((d >> 3) * 16 + att_perm(pos & 15)) * 8 + (d & 7);
}

// One workgroup per token b (it also sets the token's 16 score maxima to -1e30). q heads 0..15 and k heads 16..19 are normalised (q_norm / k_norm, sum of squares
// in fp64 in index order, one lane per head), roped on local layers (glob == 0); q stays fp32 in qkv, k and v
// go to ko[b][1024] (k | v) and to the layer's caches kc/vc [head][ctx][128] (ctx a multiple of 16) as fp16, k in att_kidx's
// blocks, v widened to fp32: f32 MFMAs and vector instructions do not issue side by side on this part (a v_cvt_f32_f16
// adds 5 cycles to a 33-cycle MFMA), and v has a conversion to an MFMA and a half. Keys widened as well cost more in bytes
// than they save in conversions (k_att_scores at 2000 tokens, global layer: 134 us against 92; k_att_pv with v in fp16
// 115 against 110). vinf[pos]: a byte per wave, set where one of the position's values is not finite.
__global__ void __launch_bounds__(256) k_qkn(float *__restrict__ qkv, int pos0, int glob, const uint16_t *__restrict__ qn,
                                             const uint16_t *__restrict__ kn, const float *__restrict__ cs,
                                             __half *__restrict__ kc, float *__restrict__ vc, uint32_t *__restrict__ vinf,
                                             __half *__restrict__ ko, float *__restrict__ mx, int ctx) {
    __shared__ float xs[20 * AT_XS];
    __shared__ float kk[20];
    int b = blockIdx.x, t = threadIdx.x, pos = pos0 + b;
    float *row = qkv + (size_t)b * AT_QKV;
    if (t < 16) mx[b * 16 + t] = -1e30f;   // the score maxima k_att_scores raises
    // every element a thread ropes has dim t % 128 (elements t + 256 m): its cos / sin pair, loaded up front
    float rc = 0.0f, rsn = 0.0f;
    if (!glob && (t & 127) < 64) {
        float2 cv = *(const float2 *)(cs + ((size_t)pos * 32 + (t & 31)) * 2);
        rc = cv.x; rsn = cv.y;
    }
    {   // all of the thread's loads first (10 q/k values, 2 v values), then the LDS and cache stores
        float qk[10], vv[2];
#pragma unroll
        for (int m = 0; m < 10; m++) qk[m] = row[t + 256 * m];
#pragma unroll
        for (int m = 0; m < 2; m++) vv[m] = row[2560 + t + 256 * m];
#pragma unroll
        for (int m = 0; m < 10; m++) { int i = t + 256 * m; xs[(i >> 7) * AT_XS + (i & 127)] = qk[m]; }
#pragma unroll
        for (int m = 0; m < 2; m++) {
            int i = t + 256 * m;
            __half h = __float2half_rn(vv[m]);
            vv[m] = __half2float(h);
            vc[((size_t)(i >> 7) * ctx + pos) * AT_HD + (i & 127)] = vv[m]; ko[(size_t)b * 1024 + 512 + i] = h;
        }
        bool bad = __ballot(!__builtin_isfinite(vv[0]) || !__builtin_isfinite(vv[1])) != 0;
        if ((t & 63) == 0) ((uint8_t *)(vinf + pos))[t >> 6] = bad;
    }
    __syncthreads();
    if (t < 20) {
        const float *x = xs + t * AT_XS;
        double ss = 0.0;
        for (int i = 0; i < AT_HD; i++) ss += (double)x[i] * (double)x[i];
        kk[t] = 1.0f / sqrtf((float)(ss / (double)AT_HD) + 1e-6f);
    }
    __syncthreads();
    float y[10];   // elements t + 256 m of the 20 heads
#pragma unroll
    for (int m = 0; m < 10; m++) {
        int i = t + m * 256, h = i >> 7, d = i & 127;
        y[m] = xs[h * AT_XS + d] * kk[h] * bf16f((h < 16 ? qn : kn)[d]);
    }
    if (!glob) {   // rope on dims 0..63 of every head: pairs (i, i + 32)
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 10; m++) { int i = t + m * 256; xs[(i >> 7) * AT_XS + (i & 127)] = y[m]; }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 10; m++) {
            int i = t + m * 256, h = i >> 7, d = i & 127;
            if (d >= 64) continue;
            if (d < 32) y[m] = __builtin_fmaf(y[m], rc, -(xs[h * AT_XS + d + 32] * rsn));
            else y[m] = __builtin_fmaf(y[m], rc, xs[h * AT_XS + d - 32] * rsn);
        }
    }
#pragma unroll
    for (int m = 0; m < 10; m++) {
        int i = t + m * 256;
        if (i < 2048) { row[i] = y[m]; continue; }
        __half hv = __float2half_rn(y[m]);
        int h = i >> 7, d = i & 127;
        kc[(size_t)(h - 16) * ctx * AT_HD + att_kidx(pos, d)] = hv; ko[(size_t)b * 1024 + i - 2048] = hv;
    }
}

// The score buffer: row (token b, head h) at (b * 16 + h) * sst, positions by their absolute index in blocks of 16, and
// inside a block position 4 i + g at 4 g + i (g, i = 0..3): the 4 values that lane group g of k_att_pv's MFMAs multiplies in
// its 4 steps are then one 16-byte word, and so are the 4 that a lane of k_att_scores' MFMAs holds. Every block that
// overlaps the window of the row's 4-token group is written whole, -inf outside the token's own window: its exp is 0
// whatever the row's maximum (at least -1e30, also where every score the token sees is -inf), and a sum or an FMA chain
// is unchanged by a zero term, exactly.
#define AT_G 4            // tokens per row tile: 4 tokens x 4 query heads = 16 MFMA rows
#define AT_LOCAL_T 576    // longest window, in whole blocks, of k_att_local: 37 KB of scores, four workgroups per CU. With 1120
                          // (two per CU) a 1024-token chunk's layers take as long as with k_att_scores and the rest, with
                          // 2200 (one) a 2048-token chunk's 1.4 times as long
// exp of x <= 0 (or -inf): dexp without its overflow check
__device__ __forceinline__ float dexp_np(float x) {
    float k = __builtin_rintf(x * 1.44269504f);
    float r = __builtin_fmaf(-k, 0.693145752f, x);
    r = __builtin_fmaf(-k, 1.42860677e-06f, r);
    float p = 1.98412698e-04f;
    p = __builtin_fmaf(p, r, 1.38888889e-03f);
    p = __builtin_fmaf(p, r, 8.33333333e-03f);
    p = __builtin_fmaf(p, r, 4.16666667e-02f);
    p = __builtin_fmaf(p, r, 1.66666667e-01f);
    p = __builtin_fmaf(p, r, 0.5f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_fmaf(p, r, 1.0f);
    p = __builtin_amdgcn_ldexpf(p, (int)k);
    return x < -104.0f ? 0.0f : p;
}

// Scores of a row tile (4 consecutive tokens x the 4 query heads of key/value head kvh) on v_mfma_f32_16x16x4_f32, which
// adds its 4 products one by one in ascending k, each as a fused multiply-add rounded to nearest (checked bit for bit on
// this part, subnormal products included): maple.c's 8 FMA lanes over the head dimension are 8 accumulators, lane j over
// dims j, j + 8, ... in order, folded by hsum8 as before. Matrix A is 16 key rows (row m = position att_perm(m) of the
// block), B the 16 query rows, held in registers. Lane (g, n) = (lane / 16, lane % 16) ends with the positions 4 i + g
// (i = 0..3) of query row n = (token n / 4, head n % 4).
struct AttRow {   // the lane's query row: its window and its 32 values, dims (4 s + g) * 8 + j
    int b, h, pb, lb; bool live;
    float q[4][8];
};
__device__ __forceinline__ void att_row(AttRow &R, const float *qkv, int b0, int nbt, int pos0, int glob, int win, int kvh, int g, int n) {
    R.b = b0 + min(n >> 2, nbt - 1); R.h = kvh * 4 + (n & 3); R.live = (n >> 2) < nbt;
    R.pb = pos0 + R.b; R.lb = att_lo(R.pb, glob, win);
    const float *qr = qkv + (size_t)R.b * AT_QKV + R.h * AT_HD;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        v4f q0 = *(const gptr_f4 *)(qr + (4 * s + g) * 8), q1 = *(const gptr_f4 *)(qr + (4 * s + g) * 8 + 4);
#pragma unroll
        for (int j = 0; j < 4; j++) { R.q[s][j] = q0[j]; R.q[s][4 + j] = q1[j]; }
    }
}
// what a tile's blocks share: its positions lo .. hi, and the run in0 .. in1 that every one of its tokens sees
struct AttTile { int lo, hi, in0, in1; };
__device__ __forceinline__ AttTile att_tile(int b0, int nbt, int pos0, int glob, int win) {
    return AttTile{att_lo(pos0 + b0, glob, win), pos0 + b0 + nbt - 1, att_lo(pos0 + b0 + nbt - 1, glob, win), pos0 + b0};
}
// lane (g, n)'s keys of block blk (att_kidx). Positions past the last one hold anything: their scores are replaced.
__device__ __forceinline__ void att_load_k(v4i *k, const __half *kc, int blk, int lane) {
    const gptr_u4 *kp = (const gptr_u4 *)(kc + (size_t)blk * AT_KBLK) + lane;
#pragma unroll
    for (int s = 0; s < 4; s++) k[s] = kp[s * 64];
}
__device__ __forceinline__ v4f att_score_block(const v4i *k, const AttRow &R, const AttTile &T, int blk, int g) {
    v4f acc[8], o;
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const __half *hh = (const __half *)&k[s];
#pragma unroll
        for (int j = 0; j < 8; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__half2float(hh[j]), R.q[s][j], acc[j], 0, 0, 0);
    }
    const float scale = 1.0f / sqrtf((float)AT_HD);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float v8[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v8[j] = acc[j][i];
        o[i] = hsum8(v8) * scale;
    }
    if (blk * 16 < T.in0 || blk * 16 + 15 > T.in1)   // uniform: some token does not see the whole block
#pragma unroll
        for (int i = 0; i < 4; i++) { int p = blk * 16 + 4 * i + g; o[i] = p >= R.lb && p <= R.pb ? o[i] : -__builtin_inff(); }
    return o;
}
// scores of blocks b, b + 4, ... below end: next(blk, o) for each; the next block's keys load during a block's MFMAs (past
// the end the last block's again: loads under a condition would be waited for at once, where the branches meet)
template <typename F>
__device__ __forceinline__ void att_scores_run(const __half *kc, const AttRow &R, const AttTile &T, int b, int end, int g, int n, F &&next) {
    v4i ka[4], kb[4];
    if (b >= end) return;
    att_load_k(ka, kc, b, g * 16 + n);
    while (true) {
        att_load_k(kb, kc, min(b + 4, end - 1), g * 16 + n);
        __builtin_amdgcn_sched_barrier(0);   // the loads ahead of the MFMAs
        next(b, att_score_block(ka, R, T, b, g));
        if ((b += 4) >= end) break;
        att_load_k(ka, kc, min(b + 4, end - 1), g * 16 + n);
        __builtin_amdgcn_sched_barrier(0);   // the loads ahead of the MFMAs
        next(b, att_score_block(kb, R, T, b, g));
        if ((b += 4) >= end) break;
    }
}
// 4 value rows x 2 dims of a lane: positions 16 blk + 4 s + g, clamped to the tile's own (a weight outside is 0; uniform
// branch: elsewhere the address is a scalar base and fixed lane offsets)
__device__ __forceinline__ void att_load_v(float2 *v, const float *vc, int blk, const AttTile &T, uint32_t lane_off, int g) {
    const char *base = (const char *)(vc + (size_t)blk * 16 * AT_HD);
    int d[4] = {0, 4 * AT_HD * 4, 8 * AT_HD * 4, 12 * AT_HD * 4};
    if (blk * 16 < T.lo || blk * 16 + 15 > T.hi)
#pragma unroll
        for (int s = 0; s < 4; s++) d[s] = (min(max(blk * 16 + 4 * s + g, T.lo), T.hi) - blk * 16 - g) * (AT_HD * 4);
#pragma unroll
    for (int s = 0; s < 4; s++) v[s] = *(const float2 *)(base + (int32_t)lane_off + d[s]);
}

// Whether the tile's zero weights (positions that not every token sees, clamped ones, the block past an odd last one) meet a
// value that is not finite. Uniform over the wave.
__device__ __forceinline__ bool att_vinf(const uint32_t *vinf, const AttTile &T, int lane) {
    int a = min(T.lo + lane, T.in0), b = min((T.in1 & ~15) + lane, T.hi);   // at most 4 and 19 positions
    return __ballot((vinf[a] | vinf[b]) != 0) != 0;
}
// acc0 / acc1 += w (A operand, row = lane % 16) x the values of block blk as the tile's tokens see them: each token runs its
// own products, with zeros for the values outside its window, and keeps the rows that are its own (lane (g, n) holds rows
// 4 g + i: token g).
__device__ __forceinline__ void att_pv_tokens(v4f &acc0, v4f &acc1, v4f w, const float2 *v, int blk, const AttTile &T, int glob, int win, int g) {
#pragma unroll 1
    for (int t = 0; t < AT_G; t++) {
        v4f a0 = acc0, a1 = acc1;
        int lo = att_lo(T.in1 + t, glob, win);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            int p = blk * 16 + 4 * s + g;
            bool in = p >= lo && p <= T.in1 + t;
            a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], in ? v[s].x : 0.0f, a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], in ? v[s].y : 0.0f, a1, 0, 0, 0);
        }
        if (g == t) { acc0 = a0; acc1 = a1; }
    }
}

// The scores of a chunk whose windows are too long for k_att_local. One wave takes blocks of 16 positions w, w + 4, ... of
// the workgroup's run (grid y; run: blocks per workgroup, a multiple of 4), the next block's keys loaded during the
// current one's MFMAs. mx is raised to the row maxima. Bound: f32 MFMA issue (75 T FMA/s on registers) plus the
// conversions and the fold. Measured at 2000 tokens from position 0, global layer: 92 us = 46 T FMA/s (vector FMAs before:
// 24 T).
__global__ void __launch_bounds__(256, 3) k_att_scores(const float *__restrict__ qkv, int nb, int pos0, int glob, int win,
                                                       const __half *__restrict__ kc, float *__restrict__ sc,
                                                       float *__restrict__ mx, int sst, int run) {
    int ntl = (nb + AT_G - 1) / AT_G, tile = ntl - 1 - (int)(blockIdx.x >> 2), kvh = blockIdx.x & 3;
    int l = threadIdx.x & 63, g = l >> 4, n = l & 15, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int b0 = tile * AT_G, nbt = min(AT_G, nb - b0);
    AttTile T = att_tile(b0, nbt, pos0, glob, win);
    kc += (size_t)kvh * sst * AT_HD;
    int blk = (T.lo >> 4) + (int)blockIdx.y * run + wv, bend = min((T.lo >> 4) + ((int)blockIdx.y + 1) * run, (T.hi >> 4) + 1);
    if (blk >= bend) return;
    AttRow R;
    att_row(R, qkv, b0, nbt, pos0, glob, win, kvh, g, n);
    float *sr = sc + (size_t)(R.b * 16 + R.h) * sst + 4 * g;
    float m = -1e30f;
    att_scores_run(kc, R, T, blk, bend, g, n, [&](int bk, v4f o) {
        m = fmaxf(fmaxf(m, fmaxf(o.x, o.y)), fmaxf(o.z, o.w));
        if (R.live) *(v4f *)(sr + bk * 16) = o;
    });
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    if (g == 0 && R.live) atomic_max_f32(mx + R.b * 16 + R.h, m);
}

// Whole attention of a row tile in one workgroup of 4 waves, for windows whose scores fit the CU's LDS several times over
// (16 rows x T positions; a 512-position window is 35 KB, four workgroups per CU): scores (each wave every 4th block of
// 16 positions) into LDS, row maxima, p = exp(s - max) in place, the sums in position order (16 lanes, one row each), then
// the weighted sum of values (wave w: dims 32 w .. +32, accumulators of even and of odd dims, since a lane's 4-byte load
// holds one of each; w = p * inv as the MFMA's A operand, 4 value rows as B). The scores never leave the CU, and p is
// formed once. While one workgroup adds its sums the others keep the matrix cores busy. Measured at 2000 tokens from
// position 0, 512-position window: 100 us (the separate kernels on MFMA: 125; on vector FMAs before: 190). ldt: LDS floats
// per row (an even number of blocks and 4 more, so the 16 rows of a 16-byte read fall in different banks).
__global__ void __launch_bounds__(256, 3) k_att_local(const float *__restrict__ qkv, int nb, int pos0, int glob, int win,
                                                      const __half *__restrict__ kc, const float *__restrict__ vc,
                                                      const uint32_t *__restrict__ vinf, float *__restrict__ att, int ldt, int sst) {
    extern __shared__ __attribute__((aligned(16))) float att_s[];
    __shared__ float red[4][16], inv_s[16];
    int ntl = (nb + AT_G - 1) / AT_G, tile = ntl - 1 - (int)(blockIdx.x >> 2), kvh = blockIdx.x & 3;
    int tid = threadIdx.x, l = tid & 63, g = l >> 4, n = l & 15, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int b0 = tile * AT_G, nbt = min(AT_G, nb - b0);
    AttTile T = att_tile(b0, nbt, pos0, glob, win);
    kc += (size_t)kvh * sst * AT_HD; vc += (size_t)kvh * sst * AT_HD;
    int bk0 = T.lo >> 4, nblk = (T.hi >> 4) + 1 - bk0;
    {
        AttRow R;
        att_row(R, qkv, b0, nbt, pos0, glob, win, kvh, g, n);
        float m = -1e30f, *sr = att_s + n * ldt + 4 * g;
        att_scores_run(kc, R, T, bk0 + wv, bk0 + nblk, g, n, [&](int bk, v4f o) {
            m = fmaxf(fmaxf(m, fmaxf(o.x, o.y)), fmaxf(o.z, o.w));
            *(v4f *)(sr + (bk - bk0) * 16) = o;
        });
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        m = fmaxf(m, __shfl_xor(m, 32, 64));
        if (g == 0) red[wv][n] = m;
    }
    __syncthreads();
    {   // 16 threads per row
        int r = tid >> 4;
        float m = fmaxf(fmaxf(red[0][r], red[1][r]), fmaxf(red[2][r], red[3][r]));
        float *q = att_s + r * ldt + (tid & 15) * 4;
        for (int k = tid & 15; k < nblk * 4; k += 16, q += 64) {
            v4f v = *(const v4f *)q;
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = dexp_np(v[i] - m);
            *(v4f *)q = v;
        }
        if ((nblk & 1) && (tid & 15) < 4) *(v4f *)(att_s + r * ldt + nblk * 16 + (tid & 15) * 4) = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    __syncthreads();
    // the first values while the sums are added
    uint32_t lo_v = (uint32_t)(g * AT_HD + wv * 32 + 2 * n) * 4;
    float2 va[4], vb[4];
    const bool vi = att_vinf(vinf, T, l);
    att_load_v(va, vc, bk0, T, lo_v, g);
    if (tid < 16) {   // in position order (4 words hold a block's positions 4 i + g)
        const float4 *q4 = (const float4 *)(att_s + tid * ldt);
        float sum = 0.0f;
        for (int k = 0; k < nblk; k++, q4 += 4) {
            float4 a = q4[0], b = q4[1], c = q4[2], d = q4[3];
            sum += a.x; sum += b.x; sum += c.x; sum += d.x; sum += a.y; sum += b.y; sum += c.y; sum += d.y;
            sum += a.z; sum += b.z; sum += c.z; sum += d.z; sum += a.w; sum += b.w; sum += c.w; sum += d.w;
        }
        inv_s[tid] = 1.0f / sum;
    }
    __syncthreads();
    const float iv = inv_s[n];
    const float *wr = att_s + n * ldt + 4 * g;
    v4f acc0 = {0.0f, 0.0f, 0.0f, 0.0f}, acc1 = acc0;
    auto block = [&](int k, const float2 *v) {
        v4f w = *(const v4f *)(wr + k * 16);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            float ws = w[s] * iv;
            acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(ws, v[s].x, acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(ws, v[s].y, acc1, 0, 0, 0);
        }
    };
    if (__builtin_expect(vi, 0))
        for (int k = 0; k < nblk; k++) {
            v4f w = *(const v4f *)(wr + k * 16) * iv;
            att_load_v(va, vc, bk0 + k, T, lo_v, g);
            att_pv_tokens(acc0, acc1, w, va, bk0 + k, T, glob, win, g);
        }
    else for (int k = 0; k < nblk; k += 2) {
        // two blocks a turn (an odd last one is followed by a block of zero weights), each one's values loaded during the
        // other's MFMAs
        att_load_v(vb, vc, bk0 + min(k + 1, nblk - 1), T, lo_v, g);
        __builtin_amdgcn_sched_barrier(0);
        block(k, va);
        att_load_v(va, vc, bk0 + min(k + 2, nblk - 1), T, lo_v, g);
        __builtin_amdgcn_sched_barrier(0);
        block(k + 1, vb);
    }
    // lane: rows 4 g + i (token g, head i), dims 32 wv + 2 n and + 1
    if (g < nbt)
#pragma unroll
        for (int i = 0; i < 4; i++)
            *(float2 *)(att + (size_t)(b0 + g) * MH + (kvh * 4 + i) * AT_HD + wv * 32 + 2 * n) = make_float2(acc0[i], acc1[i]);
}

// Softmax sums of the 16 rows (heads) of token b, one workgroup per token: p = exp(s - max) (max from
// k_att_scores), summed in position order by 16 lanes of wave 0 (one row each); inv[b * 16 + h] = 1 / sum.
// k_att_pv recomputes the same p. Waves 1-3 produce the p of 64-position chunks into two LDS buffers while
// wave 0 sums the previous chunk, and load the raw scores one chunk further ahead into registers, so the
// serial sums (the critical path) never wait for a load or an exp.
#define AT_SMCH 64
#define AT_SMPT ((16 * AT_SMCH + 191) / 192)   // p values per producer thread and chunk
__global__ void __launch_bounds__(256) k_att_softmax(int pos0, int glob, int win, const float *__restrict__ sc,
                                                     const float *__restrict__ mx, float *__restrict__ inv, int sst) {
    constexpr int LD = AT_SMCH + 4;   // 16-byte aligned rows; the 16 summing lanes hit distinct bank groups
    __shared__ __attribute__((aligned(16))) float pl[2][16 * LD];
    __shared__ float smx[16];
    int b = blockIdx.x, tid = threadIdx.x, pos = pos0 + b;
    int c16 = att_lo(pos, glob, win) & ~15, T = (pos | 15) + 1 - c16, nch = (T + AT_SMCH - 1) / AT_SMCH;   // whole blocks of 16
    const float *rows = sc + (size_t)b * 16 * sst + c16;
    const float *mr = mx + b * 16;
    int pt = tid - 64;                 // producer index (waves 1-3)
    float sv[AT_SMPT];                 // raw scores of the next chunk to produce
    auto load = [&](int c0) {
#pragma unroll
        for (int k = 0; k < AT_SMPT; k++) {
            int i = pt + 192 * k, r = i / AT_SMCH, p = i % AT_SMCH;
            sv[k] = (i < 16 * AT_SMCH && c0 + p < T) ? rows[(size_t)r * sst + c0 + p] : 0.0f;
        }
    };
    auto produce = [&](float *buf) {
#pragma unroll
        for (int k = 0; k < AT_SMPT; k++) {
            int i = pt + 192 * k;
            if (i < 16 * AT_SMCH) buf[(i / AT_SMCH) * LD + i % AT_SMCH] = dexp_np(sv[k] - smx[i / AT_SMCH]);
        }
    };
    if (tid < 16) smx[tid] = mr[tid];
    if (pt >= 0) load(0);
    __syncthreads();
    if (pt >= 0) {
        produce(pl[0]);
        if (nch > 1) load(AT_SMCH);
    }
    __syncthreads();
    float sum = 0.0f;
    for (int c = 0; c < nch; c++) {
        if (pt >= 0) {
            if (c + 1 < nch) produce(pl[(c + 1) & 1]);
            if (c + 2 < nch) load((c + 2) * AT_SMCH);
        } else if (tid < 16) {   // in position order (4 words hold a block's positions 4 i + g); read ahead of their additions
            int n = min(AT_SMCH, T - c * AT_SMCH);
            const float4 *q4 = (const float4 *)(pl[c & 1] + tid * LD);
            for (int t = 0; t < n; t += 16) {
                float4 a = q4[t / 4], bq = q4[t / 4 + 1], cq = q4[t / 4 + 2], d = q4[t / 4 + 3];
                sum += a.x; sum += bq.x; sum += cq.x; sum += d.x; sum += a.y; sum += bq.y; sum += cq.y; sum += d.y;
                sum += a.z; sum += bq.z; sum += cq.z; sum += d.z; sum += a.w; sum += bq.w; sum += cq.w; sum += d.w;
            }
        }
        __syncthreads();
    }
    if (tid < 16) inv[b * 16 + tid] = 1.0f / sum;
}

// Weighted sum of values for a row tile, tiles with the longest windows first: on v_mfma_f32_16x16x4_f32 as in
// k_att_local, so each output is maple.c's FMA chain over positions in order. The weights w = exp(s - max) * inv of 128
// positions at a time are formed by the whole workgroup into one of two LDS stages while the previous 128 are multiplied,
// their scores loaded one stage further ahead. Two row tiles per wave (a value row then feeds both) measured no faster.
__global__ void __launch_bounds__(256) k_att_pv(int nb, int pos0, int glob, int win, const float *__restrict__ sc,
                                                const float *__restrict__ mx, const float *__restrict__ inv, const float *__restrict__ vc,
                                                const uint32_t *__restrict__ vinf, float *__restrict__ att, int sst) {
    constexpr int CH = 128, LD = CH + 4, PT = 16 * CH / 4 / 256;   // PT 16-byte words of scores per thread
    __shared__ __attribute__((aligned(16))) float wl[2][16 * LD];
    int ntl = (nb + AT_G - 1) / AT_G, tile = ntl - 1 - (int)(blockIdx.x >> 2), kvh = blockIdx.x & 3;
    int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, g = l >> 4, n = l & 15;
    int b0 = tile * AT_G, nbt = min(AT_G, nb - b0);
    AttTile T = att_tile(b0, nbt, pos0, glob, win);
    vc += (size_t)kvh * sst * AT_HD;
    int c0 = T.lo & ~15, cend = (T.hi | 15) + 1, blast = T.hi >> 4;
    // staging: word k of thread tid = row (tid / 32) + 8 k, positions 4 (tid % 32) .. of the stage
    int pw = (tid & 31) * 4;
    const float *src[PT]; float mr[PT], iv[PT];
#pragma unroll
    for (int k = 0; k < PT; k++) {
        int r = (tid >> 5) + 8 * k, bt = r >> 2, rr = (b0 + min(bt, nbt - 1)) * 16 + kvh * 4 + (r & 3);
        src[k] = sc + (size_t)rr * sst + pw; mr[k] = mx[rr]; iv[k] = bt < nbt ? inv[rr] : 0.0f;
    }
    v4f raw[PT];
    auto load = [&](int p0) {   // words past the tile's last block read its first; their weights are 0
        int o = p0 + pw < cend ? p0 : c0 - pw;
#pragma unroll
        for (int k = 0; k < PT; k++) raw[k] = *(const gptr_f4 *)(src[k] + o);
    };
    auto weights = [&](int p0, float *buf) {
#pragma unroll
        for (int k = 0; k < PT; k++) {
            v4f w;
#pragma unroll
            for (int i = 0; i < 4; i++) w[i] = p0 + pw < cend ? dexp_np(raw[k][i] - mr[k]) * iv[k] : 0.0f;
            *(v4f *)(buf + ((tid >> 5) + 8 * k) * LD + pw) = w;
        }
    };
    v4f acc0 = {0.0f, 0.0f, 0.0f, 0.0f}, acc1 = acc0;
    uint32_t lo_v = (uint32_t)(g * AT_HD + wv * 32 + 2 * n) * 4;
    float2 va[4], vb[4];
    auto block = [&](const float *wr, const float2 *v) {
        v4f w = *(const v4f *)wr;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], v[s].x, acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], v[s].y, acc1, 0, 0, 0);
        }
    };
    const bool vi = att_vinf(vinf, T, l);
    if (__builtin_expect(vi, 0)) {   // token by token, stage after stage; ahead of the loop below, whose registers it would add to
        for (int p0 = c0; p0 < cend; p0 += CH) {
            __syncthreads();
            load(p0);
            weights(p0, wl[0]);
            __syncthreads();
            for (int bk = p0 >> 4; bk < min(p0 + CH, cend) >> 4; bk++) {
                att_load_v(va, vc, bk, T, lo_v, g);
                att_pv_tokens(acc0, acc1, *(const v4f *)(wl[0] + n * LD + 4 * g + (bk * 16 - p0)), va, bk, T, glob, win, g);
            }
        }
        __syncthreads();
        cend = c0;   // nothing left for the loop below
    }
    load(c0);
    att_load_v(va, vc, c0 >> 4, T, lo_v, g);
    weights(c0, wl[0]);
    if (c0 + CH < cend) load(c0 + CH);
    int st = 0;
    for (int p0 = c0; p0 < cend; p0 += CH, st ^= 1) {
        __syncthreads();   // stage st written; stage st ^ 1 no longer read
        const float *wr = wl[st] + n * LD + 4 * g;
        int bend = min(p0 + CH, cend) >> 4;   // two blocks a turn, as in k_att_local (a stage holds 8)
        for (int bk = p0 >> 4; bk < bend; bk += 2, wr += 32) {
            att_load_v(vb, vc, min(bk + 1, blast), T, lo_v, g);
            __builtin_amdgcn_sched_barrier(0);
            block(wr, va);
            att_load_v(va, vc, min(bk + 2, blast), T, lo_v, g);
            __builtin_amdgcn_sched_barrier(0);
            block(wr + 16, vb);
        }
        if (p0 + CH < cend) {
            weights(p0 + CH, wl[st ^ 1]);
            if (p0 + 2 * CH < cend) load(p0 + 2 * CH);
        }
    }
    // lane: rows 4 g + i (token g, head i), dims 32 wv + 2 n and + 1
    if (g < nbt)
#pragma unroll
        for (int i = 0; i < 4; i++)
            *(float2 *)(att + (size_t)(b0 + g) * MH + (kvh * 4 + i) * AT_HD + wv * 32 + 2 * n) = make_float2(acc0[i], acc1[i]);
}
