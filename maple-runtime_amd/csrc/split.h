// split.h -- gate/up and down in tiles of 16 pairs, each expert spread over many workgroups.
//
// With few used experts, one workgroup per expert (k_expert16) leaves most CUs idle: a CU streams about 30 GB/s, so a
// 798,720-byte expert takes 27 us however few there are. Here an expert's rows are split over 8 to 32 workgroups per
// kernel, every wave issues all of its code loads at once (16, 8 or 4 KB per gate/up wave for KS = 1, 2, 4; 4 KB per down
// wave), and act makes one trip through HBM's caches between the two launches (every row of an expert is needed before
// its act can be quantised). What bounds each kernel: the dependent loads (routing, then codes) at a few experts, the code
// stream from about a hundred. Measured against the one-workgroup kernel at the sizes where the choice between them changes: see
// split_use in mmoe.hip.
// Results are the decode kernels' bit for bit, and k_expert16's for finite inputs: the same integer sums, the same fp32
// sequence.
#pragma once
#include "kernels.h"

#define SP_MAXP 256   // pairs of one call (32 tokens): four values per lane cover a wave's copy of the top-8 lists
// Device routing: the top-8 lists in, the grouping out (what k_group publishes)
struct SplitGroup {
    const int *top; const float *tw; int nb; const ExpPtr *layer_tab; Plan *plan; Tile *tiles; ExpPtr *eptr_u; int *eu;
    int *utok; float *uw; int *tp; int *sp; int *pu; DnTile *dt;
};

// The whole grouping of maple.c:924-938 and 1018-1019 for P <= SP_MAXP pairs by one workgroup of 256 threads: counts and
// scans over the 256 experts (thread = expert), then every pair's place (thread = pair: its expert's first pair plus
// the number of earlier pairs with that expert, from the masks of pairs). lds: 12 KB of scratch.
__device__ __forceinline__ void split_publish(const SplitGroup &g, void *lds) {
    unsigned long long (*msk)[MNE] = (unsigned long long (*)[MNE])lds;   // [SP_MAXP / 64][expert]: the pairs with it
    int *ps = (int *)(msk + SP_MAXP / 64), *ux = ps + MNE, *tl = ux + MNE, (*wt)[3] = (int (*)[3])(tl + SP_MAXP);
    int t = threadIdx.x, l = t & 63, wv = t >> 6, P = g.nb * MTOPK;
    int e = t < P ? g.top[t] : -1;
    float w = t < P ? g.tw[t] : 0.0f;
    ExpPtr my = g.layer_tab[t];
#pragma unroll
    for (int k = 0; k < SP_MAXP / 64; k++) msk[k][t] = 0ull;
    tl[t] = e;
    __syncthreads();
    if (e >= 0) atomicOr(&msk[wv][e], 1ull << l);
    __syncthreads();
    int run = 0;
#pragma unroll
    for (int k = 0; k < SP_MAXP / 64; k++) run += popc64(msk[k][t]);
    int used = run > 0, nt = (run + 15) >> 4, isc = run, isu = used, ist = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int a = __shfl_up(isc, o, 64), b = __shfl_up(isu, o, 64), c = __shfl_up(ist, o, 64);
        if (l >= o) { isc += a; isu += b; ist += c; }
    }
    if (l == 63) { wt[wv][0] = isc; wt[wv][1] = isu; wt[wv][2] = ist; }
    __syncthreads();
    for (int k = 0; k < wv; k++) { isc += wt[k][0]; isu += wt[k][1]; ist += wt[k][2]; }
    int p0 = isc - run, u = isu - used, t0 = ist - nt;
    ps[t] = p0; ux[t] = u;
    g.eu[t] = used ? u : -1;
    if (used) {
        g.plan->ue[u] = t; g.plan->ustart[u] = p0; g.plan->tstart[u] = t0;
        g.eptr_u[u] = my;
        for (int i = 0; i < nt; i++) {
            int n = min(16, run - 16 * i);
            g.tiles[t0 + i] = Tile{u, p0 + 16 * i, n, 0};
            g.dt[t0 + i] = DnTile{p0 + 16 * i, n, 0, 0, my.dc, my.ds};
        }
    }
    if (t == MNE - 1) {
        g.plan->nu = isu; g.plan->np = isc; g.plan->ntile_gu = ist; g.plan->tn = 16;
        g.plan->ustart[isu] = isc; g.plan->tstart[isu] = ist;
    }
    __syncthreads();
    if (e >= 0) {
        int before = popc64(msk[wv][e] & ((1ull << l) - 1ull)), lower = 0, b = t / MTOPK;
        for (int k = 0; k < wv; k++) before += popc64(msk[k][e]);
#pragma unroll
        for (int k = 0; k < MTOPK; k++) lower += tl[b * MTOPK + k] < e;
        int pr = ps[e] + before;
        g.utok[pr] = b; g.uw[pr] = w; g.pu[pr] = ux[e]; g.sp[t] = pr; g.tp[b * MTOPK + lower] = pr;
    }
}

// Gate/up with SiLU*up of one tile (<= 16 pairs of one expert) for 64 / KS gate and up rows; block = 4 waves: wave w takes
// rows 16 (w / KS) .. +16 of both matrices and the columns of share w % KS (KS > 1: the int32 sums of the KS shares
// meet in LDS; used where the tiles alone would leave CUs idle). MFMA operands as k_gateup; the tile's n input rows in
// LDS (the others hold whatever was there: their columns are never stored). act (fp32) to HBM.
// GRP: tile = pair i's expert if i is its 1st, 17th, ... pair (else the workgroup leaves); block 0 publishes the
// grouping. grid = (P + 1) 8 KS. !GRP: tile i of the plan; grid = at least ntile 8 KS.
template <int KS, bool GRP>
__global__ void __launch_bounds__(256, 4) k_gu_split(const Plan *__restrict__ plan, const Tile *__restrict__ tiles, const ExpPtr *__restrict__ eptr,
                                                  const int *__restrict__ utok, const int8_t *__restrict__ qx,
                                                  const float *__restrict__ qsx, const int *__restrict__ qsumx,
                                                  float *__restrict__ act, int *__restrict__ dbg, SplitGroup g) {
    constexpr int NSP = 8 * KS, RW = 4 / KS, NC = 8 / KS;   // workgroups per tile, row groups, 256-column chunks per wave
    __shared__ __attribute__((aligned(16))) int8_t xs[16 * MH];
    __shared__ int toks[4][16];
    __shared__ __attribute__((aligned(16))) v4i red[KS > 1 ? 4 : 1][2][KS > 1 ? 64 : 1];
    int tid = threadIdx.x, l = tid & 63, G = l >> 4, r16 = l & 15;
    int wv = __builtin_amdgcn_readfirstlane(tid >> 6), rw = wv / KS, ks = wv % KS;
    int item = blockIdx.x / NSP, part = blockIdx.x % NSP;
    int p0, ntok;
    ExpPtr ex;
    if (GRP) {
        if (item == 0) { if (part == 0) split_publish(g, xs); return; }
        int i = item - 1, P = g.nb * MTOPK, e = g.top[i], tv[SP_MAXP / 64];
#pragma unroll
        for (int k = 0; k < SP_MAXP / 64; k++) tv[k] = k * 64 + l < P ? g.top[k * 64 + l] : 0x7fffffff;
        int less = 0, cnt = 0, rank = 0, rk[SP_MAXP / 64];
#pragma unroll
        for (int k = 0; k < SP_MAXP / 64; k++) {
            unsigned long long m = __ballot(tv[k] == e);
            less += popc64(__ballot(tv[k] < e));
            rk[k] = cnt + popc64(m & ((1ull << l) - 1ull));
            if (k * 64 <= i) rank += popc64(i - k * 64 < 64 ? m & ((1ull << (i - k * 64)) - 1ull) : m);
            cnt += popc64(m);
        }
        if (rank & 15) return;
        p0 = less + rank; ntok = min(16, cnt - rank);
        ex = g.layer_tab[e];
#pragma unroll
        for (int k = 0; k < SP_MAXP / 64; k++)
            if (tv[k] == e && rk[k] >= rank && rk[k] < rank + 16) toks[wv][rk[k] - rank] = (k * 64 + l) / MTOPK;
    } else {
        if (item >= plan->ntile_gu) return;
        Tile tl = tiles[item];
        p0 = tl.p0; ntok = tl.n;
        ex = eptr[tl.u];
        if (l < ntok) toks[wv][l] = utok[p0 + l];
    }
    int row0 = (part * RW + rw) * 16;
    uint32_t go = (uint32_t)(row0 + r16) * (MH / 4) + (G >> 1) * 32 + (G & 1) * 16 + ks * NC * 64;
    v4i cg[NC], cu[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) cg[c] = *(const gptr_u4 *)(ex.gc + go + c * 64);
#pragma unroll
    for (int c = 0; c < NC; c++) cu[c] = *(const gptr_u4 *)(ex.uc + go + c * 64);
    v4f sg = *(const gptr_f4 *)(ex.gs + row0 + 4 * G), su = *(const gptr_f4 *)(ex.us + row0 + 4 * G);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    int tr = toks[wv][min(r16, ntok - 1)];
    float qs = *(const gptr_f *)(qsx + tr);
    int qsum = *(const __attribute__((address_space(1))) int *)(qsumx + tr);
    // input rows: thread -> row 2k + tid / 128, 16-byte part tid % 128 (slot as k_gateup: part ^ row inside a chunk)
    {
        int prt = tid & 127, rh = tid >> 7;
        v4i v[8];
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (2 * k + rh < ntok) v[k] = *(const gptr_u4 *)(qx + (size_t)toks[wv][2 * k + rh] * MH + prt * 16);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            int tk = 2 * k + rh;
            if (tk < ntok) *(v4i *)(xs + tk * MH + (prt >> 4) * 256 + (((prt & 15) ^ tk) * 16)) = v[k];
        }
    }
    __syncthreads();
    v4i ag = {0, 0, 0, 0}, au = {0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < NC; c++) {
        __builtin_amdgcn_sched_barrier(0);   // decode a chunk at a time (registers: four waves per SIMD)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            int p = (G >> 1) * 8 + (G & 1) * 4 + t;
            v4i bv = *(const v4i *)(xs + r16 * MH + (ks * NC + c) * 256 + ((p ^ r16) * 16));
            uint32_t wg = (uint32_t)(t == 0 ? cg[c].x : t == 1 ? cg[c].y : t == 2 ? cg[c].z : cg[c].w);
            uint32_t wu = (uint32_t)(t == 0 ? cu[c].x : t == 1 ? cu[c].y : t == 2 ? cu[c].z : cu[c].w);
            ag = __builtin_amdgcn_mfma_i32_16x16x64_i8(decode_word(wg), bv, ag, 0, 0, 0);
            au = __builtin_amdgcn_mfma_i32_16x16x64_i8(decode_word(wu), bv, au, 0, 0, 0);
        }
    }
    if (KS > 1) {
        if (ks) { red[wv][0][l] = ag; red[wv][1][l] = au; }
        __syncthreads();
        if (ks) return;
#pragma unroll
        for (int k = 1; k < KS; k++) { ag += red[wv + k][0][l]; au += red[wv + k][1][l]; }
    }
    if (r16 >= ntok) return;
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float gv = (float)(ag[i] - qsum) * qs * sg[i];
        float uv = (float)(au[i] - qsum) * qs * su[i];
        float gg = gv < 7.0f ? gv : 7.0f;
        // maple.c's clamp of a NaN too (infinite inputs): the NaN; v_med3_f32 would make it -7
        o[i] = silu_le7(gg) * __builtin_elementwise_minimum(__builtin_elementwise_maximum(uv, -7.0f), 7.0f);
    }
    *(float4 *)(act + (size_t)(p0 + r16) * MFF + row0 + 4 * G) = make_float4(o[0], o[1], o[2], o[3]);
    if (dbg) {
        *(v4i *)(dbg + (size_t)(p0 + r16) * 2 * MFF + row0 + 4 * G) = ag;
        *(v4i *)(dbg + (size_t)(p0 + r16) * 2 * MFF + MFF + row0 + 4 * G) = au;
    }
}

// Down of one tile for 64 RF rows (wave w: RF = 2 fragments of 16): the tile's act is quantised in the workgroup while
// its codes are in flight (half-wave h takes pairs h, h + 8), D = (float)(sum - qsum) * qs * s_down[row] to HBM; the
// tile's first workgroup also writes the int8 act out. grid = at least ntile x 16. One fragment per wave (twice the
// workgroups, each quantising the tile again) takes 5.4 us against 5.6 us for 5 tokens and 8.4 against 7.4 for 12, four
// fragments 6.3 and 8.0. Tiles of 32 pairs (two token fragments here and in k_gu_split, whose workgroups then fill the LDS
// of a CU at two): 37.5 + 23.2 us at 300 tokens against 31.8 + 24.1.
__global__ void __launch_bounds__(256) k_dn_split(const Plan *__restrict__ plan, const DnTile *__restrict__ dt, const float *__restrict__ act,
                                                  int8_t *__restrict__ qa, float *__restrict__ qsa, int *__restrict__ qsuma,
                                                  float *__restrict__ down, int *__restrict__ dbg) {
    constexpr int RF = 2, NSP = 32 / RF, GS = 128, QW = MFF + 16;
    __shared__ __attribute__((aligned(16))) int8_t bs[16 * QW];
    __shared__ float sq[16];
    __shared__ int ss[16];
    int tid = threadIdx.x, l = tid & 63, G = l >> 4, r16 = l & 15, wv = tid >> 6;
    DnTile d = dt[blockIdx.x / NSP];
    if ((int)(blockIdx.x / NSP) >= plan->ntile_gu) return;
    int part = blockIdx.x % NSP, row0 = (part * 4 + wv) * RF * 16, p0 = d.p0, ntok = d.n;
    const uint8_t *cp = d.dc + (uint32_t)(row0 + r16) * (MFF / 4) + (G >> 1) * 32 + (G & 1) * 16;
    // act before the codes: loads return in issue order and the quantisation is the longer chain
    int hw = tid >> 5, o = l & 31;
    const float *ar = act + (size_t)p0 * MFF + (o >> 3) * 128 + ((o >> 2) & 1) * 16 + (o & 3) * 4;
    v4f a[2][4];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        int tk = min(hw + 8 * k, ntok - 1);
        if (k == 0 || ntok > 8)
#pragma unroll
            for (int s = 0; s < 4; s++) a[k][s] = *(const gptr_f4 *)(ar + (size_t)tk * MFF + s * 32);
    }
    v4i c[RF][2];
    v4f sd[RF];
#pragma unroll
    for (int f = 0; f < RF; f++) {
#pragma unroll
        for (int h = 0; h < 2; h++) c[f][h] = *(const gptr_u4 *)(cp + (uint32_t)f * 16 * (MFF / 4) + h * 64);
        sd[f] = *(const gptr_f4 *)(d.ds + row0 + f * 16 + 4 * G);
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
        if (k == 0 || ntok > 8) {
            float v[16];
#pragma unroll
            for (int s = 0; s < 4; s++) { v[4 * s] = a[k][s].x; v[4 * s + 1] = a[k][s].y; v[4 * s + 2] = a[k][s].z; v[4 * s + 3] = a[k][s].w; }
            int tk = hw + 8 * k;
            quant_half<GS>(v, l, bs + tk * QW, sq + tk, ss + tk);
        }
    __syncthreads();
    if (part == 0) {
        for (int i = tid; i < ntok * 32; i += 256) *(v4i *)(qa + (size_t)(p0 + (i >> 5)) * MFF + (i & 31) * 16) = *(const v4i *)(bs + (i >> 5) * QW + (i & 31) * 16);
        if (tid < ntok) { qsa[p0 + tid] = sq[tid]; qsuma[p0 + tid] = ss[tid]; }
    }
    v4i acc[RF];
#pragma unroll
    for (int f = 0; f < RF; f++) acc[f] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            v4i bv = *(const v4i *)(bs + r16 * QW + h * 256 + (G >> 1) * 128 + (G & 1) * 64 + t * 16);
#pragma unroll
            for (int f = 0; f < RF; f++) {
                const v4i cj = c[f][h];
                uint32_t w = (uint32_t)(t == 0 ? cj.x : t == 1 ? cj.y : t == 2 ? cj.z : cj.w);
                acc[f] = __builtin_amdgcn_mfma_i32_16x16x64_i8(decode_word(w), bv, acc[f], 0, 0, 0);
            }
        }
    if (r16 >= ntok) return;
    float qs = sq[r16]; int qsum = ss[r16];
    float *dp = down + (size_t)(p0 + r16) * MH;
#pragma unroll
    for (int f = 0; f < RF; f++) {
        int r = row0 + f * 16 + 4 * G;
        float ov[4];
#pragma unroll
        for (int i = 0; i < 4; i++) ov[i] = (float)(acc[f][i] - qsum) * qs * sd[f][i];
        *(float4 *)(dp + r) = make_float4(ov[0], ov[1], ov[2], ov[3]);
        if (dbg) *(v4i *)(dbg + (size_t)(p0 + r16) * MH + r) = acc[f];
    }
}
