// prefill.hip -- routed MoE FFN for a chunk of tokens (prefill): tokens are
// routed, grouped by expert, and each expert's gate/up and down projections
// run as grouped GEMMs on the matrix cores (prefill_gemm.h).  No counterpart in
// the reference, which runs its decode MoE once per prompt token
// (cs/src/qwen35_model/compute_graph.rs:1787-1800); the per-token arithmetic
// is that of cs/src/qwen35_model/moe_ffn.rs:1081-1768.
//
// Launches: P1 router logits (reference order); Q8_1(x); P2 softmax/top-k per
// token; P3 expert plan (counting sort of (token, k) pairs by expert, tiles of
// 16, 32 or 64 pairs); P4 gate/up + silu*up + Q8_1(h); P5 down; P6
// router-weighted sum in k order plus the shared expert.
#include "api_internal.h"
#include "prefill_gemm.h"

namespace chimere {

// router tile: tokens x rows per work-group (8 x 8: 100 VGPRs, four
// work-groups per CU; 16 x 8 at 170 VGPRs ran the 512-token chunk ~5 us slower)
constexpr int PF_RT = 8, PF_RE = 8;

// P1: grid (ceil((E + has_gate) / PF_RE), ceil(T / PF_RT)), 256 threads: logits
// of PF_RT tokens x PF_RE router rows.  Every output keeps the reference's order
// (elementwise.rs:186-221 launched with 256 threads): thread j accumulates
// columns j, j+256, ... with fma, then the 256 partials are summed by the
// halving tree (pairs j, j+m for m = 128, ..., 1).  Thread j owns partial j
// of all PF_RT * PF_RE outputs of the tile; the tree runs in LDS for 32 outputs at a
// time: 8 threads per output, thread q first reduces the 32 partials
// j = q (mod 8) (tree levels m = 128 .. 8), then levels 4, 2, 1 run across
// the 8 lanes.
__global__ __launch_bounds__(256) void k_pf_router(PfArgs a) {
    __shared__ float red[32][264];   // row stride = 8 banks: the 8-lane groups read distinct banks
    const int tid = threadIdx.x;
    const int NR = a.E + (a.sh_gate_w ? 1 : 0);
    // 1-D grid of ET x TT tiles.  Work-groups are dealt to the 8 XCDs
    // round-robin; when TT is a multiple of 8, XCD x takes the token tiles
    // [x TT/8, (x+1) TT/8) against every router row, so each XCD's L2 holds
    // the router once and only its own tokens' rows
    const int ET = (NR + PF_RE - 1) / PF_RE, TT = (a.T + PF_RT - 1) / PF_RT;
    int et, tt;
    if ((TT & 7) == 0) {
        const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
        tt = x * (TT >> 3) + k / ET;
        et = k - (k / ET) * ET;
    } else {
        tt = blockIdx.x / ET;
        et = blockIdx.x - tt * ET;
    }
    const int e0 = et * PF_RE, t0 = tt * PF_RT;
    const float* rows[PF_RE];
#pragma unroll
    for (int e = 0; e < PF_RE; e++) {
        const int r = min(e0 + e, NR - 1);
        rows[e] = r < a.E ? a.router + (int64_t)r * a.H : a.sh_gate_w;
    }
    float acc[PF_RT][PF_RE];
    // the loads of column step h + 256 are issued before step h's products;
    // the loop runs two column steps per trip on two register sets (no
    // copies between the sets), and every load is a uniform row base plus a
    // 32-bit lane offset (no 64-bit address arithmetic per load)
    const float* xr[PF_RT];
#pragma unroll
    for (int t = 0; t < PF_RT; t++) xr[t] = a.x + (int64_t)min(t0 + t, a.T - 1) * a.H;
    auto ld = [](const float* base, int h) {
        return *(const float*)((const char*)base + (uint32_t)h * 4u);
    };
    float r0[PF_RE], x0[PF_RT], r1[PF_RE], x1[PF_RT];
    auto load = [&](float (&r)[PF_RE], float (&x)[PF_RT], int h) {
#pragma unroll
        for (int e = 0; e < PF_RE; e++) r[e] = ld(rows[e], h);
#pragma unroll
        for (int t = 0; t < PF_RT; t++) x[t] = ld(xr[t], h);
    };
    auto step = [&](const float (&r)[PF_RE], const float (&x)[PF_RT]) {
#pragma unroll
        for (int t = 0; t < PF_RT; t++)
#pragma unroll
            for (int e = 0; e < PF_RE; e++) acc[t][e] = __builtin_fmaf(r[e], x[t], acc[t][e]);
    };
    // column step tid (acc = fmaf(r, x, 0), the first fma of the chain)
    load(r0, x0, tid);
    load(r1, x1, tid + 256 < a.H ? tid + 256 : tid);
#pragma unroll
    for (int t = 0; t < PF_RT; t++)
#pragma unroll
        for (int e = 0; e < PF_RE; e++) acc[t][e] = __builtin_fmaf(r0[e], x0[t], 0.0f);
    // h: the step whose operands are in set 1 (H is a multiple of 256, so
    // every bound below is uniform)
    for (int h = tid + 256; h < a.H; h += 512) {
        load(r0, x0, h + 256 < a.H ? h + 256 : h);
        step(r1, x1);
        if (h + 256 >= a.H) break;
        load(r1, x1, h + 512 < a.H ? h + 512 : h);
        step(r0, x0);
    }
    const int o = tid >> 3, q = tid & 7;
#pragma unroll
    for (int rnd = 0; rnd < PF_RT * PF_RE / 32; rnd++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const int oo = rnd * 32 + i;
            red[i][tid] = acc[oo / PF_RE][oo % PF_RE];
        }
        __syncthreads();
        float v[32];
#pragma unroll
        for (int i = 0; i < 32; i++) v[i] = red[o][q + 8 * i];
#pragma unroll
        for (int m = 16; m >= 1; m >>= 1)
#pragma unroll
            for (int i = 0; i < m; i++) v[i] = v[i] + v[i + m];
        float w = v[0];
        w = w + xlane<4>(w);
        w = w + xlane<2>(w);
        w = w + xlane<1>(w);
        const int oo = rnd * 32 + o, t = t0 + oo / PF_RE, e = e0 + oo % PF_RE;
        if (q == 0 && t < a.T && e < NR) {
            if (e < a.E) a.logits[(int64_t)t * a.E + e] = a.bias ? w + a.bias[e] : w;
            else a.glogit[t] = w;
        }
    }
}

// Q8_1 of x (the values of k_quantize_q8_1) in the GEMMs' layout.  Eight lanes per block, 16-byte loads
// (two half-waves per block with 4-byte loads and 2-byte stores: 4096 tokens
// 19.7 us).  Grid: groups of 32 blocks of all tokens
__global__ __launch_bounds__(256) void k_pf_quant(PfArgs a) {
    const int64_t b = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
    const int i = threadIdx.x & 7;
    if (b >= (int64_t)a.T * (a.H / QK)) return;   // whole groups of eight lanes exit together
    const float* src = a.x + b * QK + 4 * i;
    float v[4];
    if (((uintptr_t)a.x & 15) == 0) {
        const float4 u = *(const float4*)src;
        v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = src[k];
    }
    float amax = __builtin_fabsf(v[0]);
#pragma unroll
    for (int k = 1; k < 4; k++) amax = __builtin_fmaxf(amax, __builtin_fabsf(v[k]));
    amax = __builtin_fmaxf(amax, xlane<4>(amax));
    amax = __builtin_fmaxf(amax, xlane<2>(amax));
    amax = __builtin_fmaxf(amax, xlane<1>(amax));
    const float d = amax / 127.0f;
    v4h h;
    int sq = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        // (int8_t): where d underflows to 0 the byte the Q8_1 block would hold
        const int q = amax == 0.0f ? 0 : (int8_t)(int)__builtin_roundf(v[k] / d);
        h[k] = (_Float16)q;
        sq += q;
    }
    sq += xlane<4>(sq);
    sq += xlane<2>(sq);
    sq += xlane<1>(sq);
    *(v4h*)(a.xh + b * QK + 4 * i) = h;
    if (i == 0) {
        const uint32_t dh = f2h(d);
        a.xd[b] = dh;
        a.xs[b] = h2f(dh) * (float)sq;   // exact: 11 x 12 bits
    }
}

// P2: one wave per token, 16 tokens per work-group; each pair's rank among the
// work-group's pairs of its expert, and the work-group's count of every expert
// (counted in global memory instead, the returning atomics of 4096 tokens took
// 15 us)
constexpr int PF_TKT = 16;
__global__ __launch_bounds__(64 * PF_TKT) void k_pf_topk(PfArgs a) {
    __shared__ uint64_t s_tk[PF_TKT][128];
    __shared__ int s_ids[PF_TKT][MAX_K], cnt[MAX_E];
    __shared__ float s_w[PF_TKT][MAX_K];
    const int tid = threadIdx.x, wave = tid >> 6, t = blockIdx.x * PF_TKT + wave;
    for (int e = tid; e < a.E; e += 64 * PF_TKT) cnt[e] = 0;
    if (t < a.T) topk_wave_any(a.logits + (int64_t)t * a.E, a.E, a.K, s_ids[wave], s_w[wave], s_tk[wave]);
    __syncthreads();
    // thread -> pair of the work-group (16 tokens x at most 16 experts)
    const int pt = tid / MAX_K, k = tid - pt * MAX_K;
    const bool on = pt < PF_TKT && k < a.K && blockIdx.x * PF_TKT + pt < a.T;
    int e = -1, r = 0;
    if (on) {
        e = s_ids[pt][k];
        if ((unsigned)e < (unsigned)a.E) r = atomicAdd(&cnt[e], 1);
        else e = -1;
    }
    if (on) {
        const int64_t p = (int64_t)(blockIdx.x * PF_TKT + pt) * a.K + k;
        a.ids[p] = e;
        a.wts[p] = s_w[pt][k];
        a.rank[p] = r;
    }
    __syncthreads();
    for (int i = tid; i < a.E; i += 64 * PF_TKT) a.cnt[(int64_t)blockIdx.x * a.E + i] = cnt[i];
}

// exclusive prefix sum of one int per thread over a 1024-thread group
__device__ __forceinline__ int excl_scan1024(int v, int* wsum, int* total) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    if (w == 0) {
        const int t = lane < 16 ? wsum[lane] : 0;
        int sc = t;
#pragma unroll
        for (int d = 1; d < 16; d <<= 1) {
            const int y = __shfl_up(sc, d);
            if (lane >= d) sc += y;
        }
        __syncthreads();   // pairs with the barrier below for the other waves
        if (lane < 16) wsum[lane] = sc - t;
        if (lane == 15) *total = sc;
    } else {
        __syncthreads();
    }
    __syncthreads();
    return x - v + wsum[w];
}

// P3: counting sort of the T*K pairs by expert (inside an expert by 16-token top-k
// work-group, otherwise in any order, which may differ between runs: every
// pair's output row is computed on its own, so no result depends on it), the shared expert as expert E with all T
// tokens, and the list of tiles of up to tile_pairs pairs.  Every work-group
// sums the counts of all top-k work-groups (each expert's total, and what comes
// before its own PF_PLG of them), scans the totals (thread i: experts 2i and
// 2i+1) and places its pairs; the first one also writes the tiles.  (One
// work-group counting and placing all pairs: 4096 tokens top-8 40 us.)
constexpr int PF_PLG = 4;   // top-k work-groups (64 tokens, at most 1024 pairs) per plan work-group
__global__ __launch_bounds__(1024) void k_pf_plan(PfArgs a) {
    __shared__ int first[1024], total[1024], before[1024];
    __shared__ int wsum[16], tot[2];
    const int tid = threadIdx.x, TK = a.T * a.K, E = a.E, TP = a.tile_pairs;
    const int ntk = (a.T + PF_TKT - 1) / PF_TKT, g0 = blockIdx.x * PF_PLG;
    const int p0 = blockIdx.x * PF_PLG * PF_TKT * a.K, np = min(TK - p0, PF_PLG * PF_TKT * a.K);
    const int e = tid < np ? a.ids[p0 + tid] : -1;
    const int rank = tid < np ? a.rank[p0 + tid] : 0;
    if (blockIdx.x == 0 && a.whole)
        for (int i = tid; i < 8 * (pf_eighth(a.nsh) + pf_eighth(a.max_tiles)); i += 1024)
            a.tiles[i] = make_int4(0, 0, 0, 0);
    total[tid] = 0;
    before[tid] = 0;
    __syncthreads();
    {
        // 1024 / EP threads per expert, each over every (1024 / EP)-th top-k work-group
        const int EP = E <= 256 ? 256 : E <= 512 ? 512 : 1024, seg = tid / EP, nseg = 1024 / EP, ex = tid - seg * EP;
        if (ex < E) {
            int s = 0, sb = 0;
#pragma unroll 8
            for (int g = seg; g < ntk; g += nseg) {
                const int c = a.cnt[(int64_t)g * E + ex];
                s += c;
                sb += g < g0 ? c : 0;
            }
            atomicAdd(&total[ex], s);
            atomicAdd(&before[ex], sb);
        }
    }
    __syncthreads();
    const int c0 = tid < 512 ? total[2 * tid] : 0, c1 = tid < 512 ? total[2 * tid + 1] : 0;
    const int po = excl_scan1024(c0 + c1, wsum, &tot[0]);
    if (tid < 512) {
        first[2 * tid] = po;
        first[2 * tid + 1] = po + c0;
    }
    __syncthreads();
    if (e >= 0) {
        // the pair's top-k work-group is g0 + tid / (16 K): the counts of the
        // plan work-group's earlier ones come before it too
        int pos = first[e] + before[e] + rank;
        for (int g = g0; g < g0 + tid / (PF_TKT * a.K); g++) pos += a.cnt[(int64_t)g * E + e];
        const int p = p0 + tid;
        a.spairs[pos] = p;
        a.stok[pos] = p / a.K;
        if (a.ids_out) { a.ids_out[p] = e; a.w_out[p] = a.wts[p]; }
    }
    const int t0 = blockIdx.x * PF_PLG * PF_TKT;
    if (a.has_shared && tid < PF_PLG * PF_TKT && t0 + tid < a.T) {
        a.spairs[tot[0] + t0 + tid] = TK + t0 + tid;
        a.stok[tot[0] + t0 + tid] = t0 + tid;
    }
    if (blockIdx.x != 0) return;
    // the tile list, arranged for pf_place
    const int n0 = (c0 + TP - 1) / TP, n1 = (c1 + TP - 1) / TP, nsh = a.nsh;
    const int to = excl_scan1024(n0 + n1, wsum, &tot[1]);
    const int per = max(pf_eighth(tot[1]), 1), persh = pf_eighth(nsh);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int c = h ? c1 : c0, base = h ? po + c0 : po, tb = h ? to + n0 : to;
        for (int s = 0; s * TP < c; s++) {
            const int t = tb + s, x = t / per;
            a.tiles[a.whole ? 8 * (persh + t - x * per) + x : 1 + nsh + t] =
                make_int4(2 * tid + h, base + s * TP, min(TP, c - s * TP), 0);
        }
    }
    for (int s = tid; s < nsh; s += 1024)
        a.tiles[a.whole ? s : 1 + s] = make_int4(E, tot[0] + s * TP, min(TP, a.T - s * TP), 0);
    if (tid == 0 && !a.whole) a.tiles[0] = make_int4(tot[1], 0, 0, 0);
}

// P6: grid (ceil(H/256), T): out = sum_k fmaf(w_k, dn_k, acc) (+ shared expert)
// one thread per 4 consecutive outputs of a token (H % 4 == 0, which every
// shape the prefill accepts has: H is a multiple of 256); each output's
// fmaf chain over k is the one of the decode layer's combine
__global__ __launch_bounds__(256) void k_pf_combine(PfArgs a) {
    const int t = blockIdx.y, h = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (h >= a.H) return;
    float4 v[MAX_K + 1];
#pragma unroll
    for (int k = 0; k < MAX_K; k++)
        if (k < a.K) v[k] = *(const float4*)(a.dn + (int64_t)(t * a.K + k) * a.H + h);
    if (a.has_shared) v[MAX_K] = *(const float4*)(a.dn + (int64_t)(a.T * a.K + t) * a.H + h);
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < MAX_K; k++) {
        if (k < a.K) {
            const float w = a.wts[t * a.K + k];
            acc.x = __builtin_fmaf(w, v[k].x, acc.x);
            acc.y = __builtin_fmaf(w, v[k].y, acc.y);
            acc.z = __builtin_fmaf(w, v[k].z, acc.z);
            acc.w = __builtin_fmaf(w, v[k].w, acc.w);
        }
    }
    float4 o = acc;
    if (a.has_shared) {
        const float4 shv = v[MAX_K];
        if (a.sh_gate_w) {
            const float sg = 1.0f / (1.0f + det_exp(-a.glogit[t]));
            o = make_float4(__builtin_fmaf(shv.x, sg, acc.x), __builtin_fmaf(shv.y, sg, acc.y),
                            __builtin_fmaf(shv.z, sg, acc.z), __builtin_fmaf(shv.w, sg, acc.w));
        } else {
            o = make_float4(shv.x + acc.x, shv.y + acc.y, shv.z + acc.z, shv.w + acc.w);
        }
    }
    float* dst = a.out + (int64_t)t * a.H + h;
    if (((uintptr_t)a.out & 15) == 0) {
        *(float4*)dst = o;
    } else {   // a caller's output that is not 16-byte aligned
        dst[0] = o.x; dst[1] = o.y; dst[2] = o.z; dst[3] = o.w;
    }
}

struct PfPlan {
    size_t logits, glogit, ids, wts, cnt, rank, spairs, stok, tiles, dn, xh, xd, xs, hh, hd, hs, total;
    int tile_pairs, nsh, max_tiles, whole, dn_ns;
};

static size_t al256p(size_t n) { return (n + 255) & ~(size_t)255; }

// Pairs per GEMM tile, by the average pairs per expert: a weight block is
// decoded once per tile, so a tile should hold an expert's pairs, but a wider
// tile's LDS and registers leave two work-groups per CU instead of three.
// Of 32 pairs and 64, the wider tile decodes fewer blocks but has a short tile
// per expert; it gains earlier with Q8_0 experts (more bytes per block).
// Chunk, 16 / 32 / 64 pairs (us), H = 2048, F = 512, 256 experts, top-8, by average:
//   IQ3_S + Q5_K  11 190 / 197 / 218   13 205 / 203 / 221   15 224 / 213 / 226
//                 24 308 / 249 / 252   28 339 / 278 / 276   32 371 / 311 / 298
//   Q4_0          11 174 / 180 / 198   13 185 / 183 / 203   24 267 / 228 / 229
//                 28 291 / 248 / 250   32 318 / 274 / 269
//   Q8_0          11 256 / 253 / 264   13 266 / 257 / 270   20 332 / 280 / 289
//                 22 343 / 287 / 293   24 358 / 309 / 300   28 386 / 330 / 314
// H = F = 1024, 64 experts, top-4: IQ3_S + Q5_K 13 76 / 79 / 92, 17 93 / 89 / 95, 28
// 115 / 98 / 104; H = 2048, F = 768, 16 experts, top-2: 20 65 / 73 / 86, 40 94 / 86 / 89.
// Skewed (logits lowered by the log of the expert's rank), IQ3_S + Q5_K: 8 138 / 123 /
// 137, 13 187 / 157 / 178, 20 249 / 207 / 215, 35 395 / 313 / 311: the average understates
// the experts that most pairs meet (Q8_0 20 290 / 232 / 218).
static int pf_tile_pairs(int te, int E, int K, int T) {
    const double avg = (double)T * K / E;
    return avg <= 13 ? PF_PT : avg <= (te == T_Q8_0 ? 20 : 28) ? 2 * PF_PT : 4 * PF_PT;
}

// The experts' tiles (at most) from which whole tiles are dealt to the XCDs
// (by whole tiles an XCD has at most 12 / tiles more than the average).  Whole /
// slices (us), H = 2048, F = 512, 256 experts, top-8: 343 tiles IQ3_S + Q5_K 248 / 243;
// 384 Q4_0 193.1 / 193.6; 408 Q4_0 + Q6_K 235 / 223, IQ3_S + Q5_K 239 / 228, Q4_0
// 205 / 209; 464 IQ3_S + Q5_K 216 / 218, Q4_0 186 / 189, Q4_0 + Q6_K 195 / 199; 768
// IQ3_S + Q5_K 808 / 822, Q4_0 733 / 747
constexpr int PF_WHOLE_TILES = 384;
// Work-groups that the down launch would have at most (the tiles' bound) with two
// slices each, up to which it takes one: two leave CUs idle behind the longest
// chain of slices.  Chunk with two / one (us): H = F = 1024, 32 experts, top-2,
// 12 tokens (104) IQ3_S + Q5_K 53 / 44, Q8_0 49 / 42, 1000 tokens (188) IQ3_S + Q5_K
// 129 / 109; H = 4096, F = 1024, 64 experts, top-4, 100 tokens (1536) Q8_0 238 / 232,
// 200 tokens (2032) 273 / 268; H = 2048, F = 512, 256 experts, top-8, 16 tokens
// (1096) 110 / 107, 64 tokens (2336) Q8_0 187 / 185 but IQ3_S + Q5_K 132 / 134,
// 512 tokens (3200) 212 / 216, Q4_0 195 / 199.  Rows of one K chunk (F = 256) are all
// start: H = 1024, 64 experts, top-6, 500 tokens (472) IQ3_S + Q5_K 70.5 / 66.3, Q8_0
// 63.7 / 64.8, 1500 tokens (912) 110.7 / 111.7, 103.8 / 105.2.
constexpr int PF_DN_ONE = 2048, PF_DN_ONE_K8 = 512;

static PfPlan plan_pf(int te, int H, int F, int E, int K, int T) {
    PfPlan p{};
    size_t o = 0;
    const size_t P = (size_t)T * K + T;
    p.tile_pairs = pf_tile_pairs(te, E, K, T);
    // an expert of c pairs has at most c / tile_pairs + 1 tiles
    auto tiles = [&](int tp) { return T * K / tp + (T * K < E ? T * K : E); };
    p.max_tiles = tiles(p.tile_pairs);
    p.nsh = (T + p.tile_pairs - 1) / p.tile_pairs;
    p.whole = p.max_tiles >= PF_WHOLE_TILES;
    p.dn_ns = (int64_t)(p.max_tiles + p.nsh) * (H / (2 * PF_ROWS)) <= (F > 256 ? PF_DN_ONE : PF_DN_ONE_K8) ? 1 : 2;
    auto take = [&](size_t& at, size_t bytes) { at = o; o += al256p(bytes); };
    take(p.logits, (size_t)T * E * 4);
    take(p.glogit, (size_t)T * 4);
    take(p.ids, (size_t)T * K * 4);
    take(p.wts, (size_t)T * K * 4);
    take(p.cnt, (size_t)((T + PF_TKT - 1) / PF_TKT) * E * 4);
    take(p.rank, (size_t)T * K * 4);
    take(p.spairs, P * 4);
    take(p.stok, P * 4);
    take(p.tiles, (size_t)(tiles(PF_PT) + (T + PF_PT - 1) / PF_PT + 16) * sizeof(int4));
    take(p.dn, P * H * 4);
    take(p.xh, (size_t)T * H * 2);
    take(p.xd, (size_t)T * (H / QK) * 4);
    take(p.xs, (size_t)T * (H / QK) * 4);
    take(p.hh, P * F * 2);
    take(p.hd, P * (F / QK) * 4);
    take(p.hs, P * (F / QK) * 4);
    p.total = o;
    return p;
}

static void launch_pf(const PfArgs& a, int te, int ts, hipStream_t s) {
    hipLaunchKernelGGL(k_pf_router,
                       dim3(((a.E + (a.sh_gate_w ? 1 : 0) + PF_RE - 1) / PF_RE) * ((a.T + PF_RT - 1) / PF_RT)),
                       dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_pf_quant, dim3((unsigned)(((int64_t)a.T * (a.H / QK) + 31) / 32)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_pf_topk, dim3((a.T + PF_TKT - 1) / PF_TKT), dim3(64 * PF_TKT), 0, s, a);
    hipLaunchKernelGGL(k_pf_plan, dim3((a.T + PF_PLG * PF_TKT - 1) / (PF_PLG * PF_TKT)), dim3(1024), 0, s, a);
    if (te == T_Q4_0) pf_launch_experts<T_Q4_0>(a, ts, s);
    else if (te == T_Q8_0) pf_launch_experts<T_Q8_0>(a, ts, s);
    else pf_launch_experts<T_IQ3_S>(a, ts, s);
    hipLaunchKernelGGL(k_pf_combine, dim3((a.H / 4 + 255) / 256, a.T), dim3(256), 0, s, a);
}

}  // namespace chimere

using namespace chimere;

extern "C" {

size_t chimere_moe_prefill_workspace_size(const chimere_moe_layer* L, int max_ntok) {
    if (!L || max_ntok < 1) return 0;
    return plan_pf(L->expert_type, L->hidden, L->ffn, L->n_experts, L->top_k, max_ntok).total;
}

void chimere_moe_prefill(const chimere_moe_layer* L, const float* x, float* out, int ntok, int* ids_out,
                         float* w_out, void* workspace, size_t ws_bytes, hipStream_t stream) {
    CHIMERE_REQUIRE(L && x && out && workspace, CHIMERE_ERR_ARG, "moe_prefill: null pointer");
    const int H = L->hidden, F = L->ffn, E = L->n_experts, K = L->top_k;
    CHIMERE_REQUIRE(ntok >= 1, CHIMERE_ERR_ARG, "moe_prefill: ntok=%d", ntok);
    CHIMERE_REQUIRE(H > 0 && H % 256 == 0 && F > 0 && F % 256 == 0, CHIMERE_ERR_ARG,
                    "moe_prefill: hidden=%d / ffn=%d must be multiples of 256", H, F);
    CHIMERE_REQUIRE(E >= 1 && E <= MAX_E && K >= 1 && K <= MAX_K && K <= E, CHIMERE_ERR_ARG,
                    "moe_prefill: n_experts=%d top_k=%d out of range", E, K);
    const bool has_sh = L->shared_type >= 0;
    auto pf_type = [](int t) { return t == T_Q4_0 || t == T_Q8_0 || t == T_IQ3_S; };
    CHIMERE_REQUIRE(pf_type(L->expert_type) &&
                        (!has_sh || pf_type(L->shared_type) || L->shared_type == T_Q4_K || L->shared_type == T_Q5_K ||
                         L->shared_type == T_Q6_K),
                    CHIMERE_ERR_ARG,
                    "moe_prefill: Q4_0 / Q8_0 / IQ3_S experts, shared expert also Q4_K / Q5_K / Q6_K (expert %d, shared %d)",
                    L->expert_type, L->shared_type);
    CHIMERE_REQUIRE(!has_sh || (L->sh_gate && L->sh_up && L->sh_down), CHIMERE_ERR_ARG,
                    "moe_prefill: shared expert incomplete");
    CHIMERE_REQUIRE(L->router_w && L->gate_exps && L->up_exps && L->down_exps, CHIMERE_ERR_ARG,
                    "moe_prefill: null weight pointer");
    CHIMERE_REQUIRE(!ids_out == !w_out, CHIMERE_ERR_ARG, "moe_prefill: ids_out and w_out go together");
    const int64_t rbH = row_bytes(L->expert_type, H), rbF = row_bytes(L->expert_type, F);
    CHIMERE_REQUIRE(L->gate_stride >= rbH * F && L->up_stride >= rbH * F && L->down_stride >= rbF * H,
                    CHIMERE_ERR_ARG, "moe_prefill: expert strides too small");
    CHIMERE_REQUIRE((((uintptr_t)L->gate_exps | (uintptr_t)L->up_exps | (uintptr_t)L->down_exps |
                      (uintptr_t)L->gate_stride | (uintptr_t)L->up_stride | (uintptr_t)L->down_stride) & 1) == 0,
                    CHIMERE_ERR_ARG, "moe_prefill: weights must be 2-byte aligned");
    const PfPlan p = plan_pf(L->expert_type, H, F, E, K, ntok);
    CHIMERE_REQUIRE(ws_bytes >= p.total && ((uintptr_t)workspace & 255) == 0, CHIMERE_ERR_WORKSPACE,
                    "moe_prefill: workspace %zu bytes < %zu (or not 256-byte aligned)", ws_bytes, p.total);
    uint8_t* w = (uint8_t*)workspace;
    PfArgs a{};
    a.H = H; a.F = F; a.E = E; a.K = K; a.T = ntok; a.has_shared = has_sh;
    a.x = x; a.out = out; a.router = L->router_w; a.bias = L->logit_bias;
    a.gate = (const uint8_t*)L->gate_exps; a.up = (const uint8_t*)L->up_exps; a.down = (const uint8_t*)L->down_exps;
    a.sg = L->gate_stride; a.su = L->up_stride; a.sd = L->down_stride;
    a.sh_gate = (const uint8_t*)L->sh_gate; a.sh_up = (const uint8_t*)L->sh_up; a.sh_down = (const uint8_t*)L->sh_down;
    a.sh_gate_w = has_sh ? L->sh_gate_w : nullptr;
    a.ids_out = ids_out; a.w_out = w_out;
    a.logits = (float*)(w + p.logits); a.glogit = (float*)(w + p.glogit);
    a.ids = (int*)(w + p.ids); a.wts = (float*)(w + p.wts);
    a.cnt = (int*)(w + p.cnt); a.rank = (int*)(w + p.rank);
    a.spairs = (int*)(w + p.spairs);
    a.stok = (int*)(w + p.stok); a.tiles = (int4*)(w + p.tiles);
    a.dn = (float*)(w + p.dn);
    a.xh = (_Float16*)(w + p.xh); a.xd = (uint32_t*)(w + p.xd); a.xs = (float*)(w + p.xs);
    a.hh = (_Float16*)(w + p.hh); a.hd = (uint32_t*)(w + p.hd); a.hs = (float*)(w + p.hs);
    a.tile_pairs = p.tile_pairs; a.nsh = has_sh ? p.nsh : 0; a.max_tiles = p.max_tiles; a.whole = p.whole;
    a.dn_ns = p.dn_ns;
    launch_pf(a, L->expert_type, has_sh ? L->shared_type : L->expert_type, stream);
    check_launch("moe_prefill");
}

}  // extern "C"
