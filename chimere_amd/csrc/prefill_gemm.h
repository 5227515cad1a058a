// prefill_gemm.h -- the expert projections of the prefill chunk (prefill.hip):
// grouped GEMMs on the matrix cores over GGUF weight blocks and activations
// quantized as Q8_1 blocks.  Instantiated per expert type in
// prefill_gemm_*.hip.
//
// Arithmetic (the L = 1 order): per output and 32-element block, ascending,
//   acc = fmaf(f32(d_w) * f32(d_x), (float)sumi, acc),
// sumi the exact integer dot of the block's quants.  Both factors come from
// the matrix cores, so that the vector ALU has one fma per output and block:
//  * sumi by v_mfma_f32_16x16x32_f16 on the quants as f16 (weights times
//    their integer sub-block scale): every product and partial sum is an
//    integer below 2^24, so the f32 result is the exact integer, already a
//    float;
//  * the scale products by v_mfma_f32_16x16x4_4b_f16, four rank-1 products
//    per instruction (three of its four terms zero; a product of two f16
//    values, subnormal ones too, is exact in f32).  Measured: it holds up the
//    vector ALU for 6 cycles, the f32 form (which runs on it) for 38, the 16
//    multiplies for 67.
// The int8 product + int -> float conversion + multiply + fma of one output
// and block on the vector ALU were 12 of 24 VALU instructions per 16x16x32
// product (512 tokens, Q4_0).
#pragma once
#include "common.h"
#include "moe_common.h"

namespace chimere {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int PF_PT = 16;        // (token, k) pairs per 16-row matrix tile
constexpr int PF_THREADS = 256;  // 4 waves

struct PfArgs {
    int H, F, E, K, T, has_shared;
    const float* x;
    float* out;
    const float* router;
    const float* bias;
    const uint8_t *gate, *up, *down;
    int64_t sg, su, sd;
    const uint8_t *sh_gate, *sh_up, *sh_down;
    const float* sh_gate_w;
    int* ids_out;
    float* w_out;
    // workspace
    float* logits;   // [T][E]
    float* glogit;   // [T]
    int* ids;        // [T*K]
    float* wts;      // [T*K]
    int* cnt;        // [top-k work-groups][E] pairs of each expert
    int* rank;       // [T*K] a pair's place among its expert's of its top-k work-group
    int* spairs;     // [T*K + T] pairs grouped by expert (shared expert last)
    int* stok;       // [T*K + T] the pairs' tokens, in the same order
    int4* tiles;     // (expert, first position in spairs, pairs or 0) of each tile, arranged for pf_place
    float* dn;       // [T*K + T][H] down-projection output per pair
    // Q8_1 blocks of x (by token) and of h (by position in spairs) as the
    // GEMMs read them: the quants as f16, the block's f16 scale in the low
    // half of a word, and (for the K-quants' min terms) that scale times the sum of
    // its quants, exact in f32
    _Float16 *xh, *hh;
    uint32_t *xd, *hd;
    float *xs, *hs;
    int tile_pairs;   // most pairs per tile: PF_PT * MT of the GEMM launches
    int nsh;          // tiles of the shared expert
    int max_tiles;    // most tiles of the experts
    int whole;        // whole tiles are dealt to the XCDs (pf_place)
    int dn_ns;        // 128-row slices per work-group of the down launch: 1 or 2
};

// ---- a weight row's chunk in LDS

// 32-element blocks per chunk: 8 (the 256-element types' superblock), Q8_0 4
// (its 34-byte blocks)
template <int T>
constexpr int pf_ch() { return T == T_Q8_0 ? 4 : 8; }
// bytes of a chunk
template <int T>
constexpr int pf_cb() { return QTraits<T>::ELEMS == 256 ? QTraits<T>::BYTES : pf_ch<T>() * QTraits<T>::BYTES; }
// 16-byte slots of an LDS row: the aligned span that holds a chunk starting at
// any even address (up to 14 bytes into its first granule)
template <int T>
constexpr int pf_sl() { return (pf_cb<T>() + 14 + 15) / 16 + (T == T_IQ3_S || T == T_Q6_K || T == T_Q5_K ? 1 : 0); }
// LDS offset of row r.  An odd number of slots starts 8 consecutive rows in
// different eighths of the banks (IQ3_S 9, Q6_K 15, Q5_K 13); 10 slots (Q4_0, Q8_0, Q4_K) do
// with one slot more after every fourth row.  (The gate/up profiles still count 0.44 of
// the LDS cycles in conflict with Q4_0, 0.54 with IQ3_S; besides the codebook
// lookups it is not known which reads these are.)
template <int T>
constexpr bool pf_skew() { return pf_sl<T>() % 2 == 0; }
template <int T>
__host__ __device__ constexpr int pf_row(int r) { return (r * pf_sl<T>() + (pf_skew<T>() ? r >> 2 : 0)) * 16; }
constexpr int PF_ROWS = 128;     // weight rows of a work-group: two groups of 64, 16 + 16 per wave
// bytes of a stage (16: the word reads of the last row)
template <int T>
constexpr int pf_wst() { return pf_row<T>(PF_ROWS) + 16; }

template <int T>
constexpr bool pf_kq() { return T == T_Q4_K || T == T_Q5_K; }

// IQ3_S codebook as f16: entry i = four levels in {1, 3, ..., 15}
struct Iq3sHalfGrid {
    uint32_t w[1024];
    static constexpr uint32_t f16_of(uint32_t v) {   // 1 <= v < 2048
        int e = 0;
        while ((v >> (e + 1)) != 0) e++;
        return (uint32_t)(15 + e) << 10 | ((v << (10 - e)) & 0x3FFu);
    }
    constexpr Iq3sHalfGrid() : w() {
        constexpr uint32_t base[512] = CHIMERE_IQ3S_GRID_INIT;
        for (int i = 0; i < 512; i++)
            for (int k = 0; k < 2; k++)
                w[2 * i + k] = f16_of((base[i] >> (16 * k)) & 0xFFu) | f16_of((base[i] >> (16 * k + 8)) & 0xFFu) << 16;
    }
};
static __device__ const Iq3sHalfGrid c_iq3s_hgrid{};

// bytes of lo, hi (elements 0..3, 4..7) as f16 1024 + byte
__device__ __forceinline__ v8h pf_bytes_h(uint32_t lo, uint32_t hi) {
    const uint4 r = make_uint4(__builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u),
                               __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u),
                               __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u),
                               __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u));
    return __builtin_bit_cast(v8h, r);
}

// One lane's view of its row's chunk: lane group q (0..3) supplies elements
// 8q .. 8q+7 of each block.  begin(): once per chunk, `s` the row's start in
// LDS (even).  The elements of block b (a compile-time value after unrolling)
// come in three steps, so that the GEMM can run them some blocks ahead:
// load() issues the LDS reads, look() the codebook lookups (IQ3_S), frag()
// gives the f16 integers (the sub-block scale multiplied in).  dw(b): the
// block's f16 scale, b per lane.
template <int T> struct PfRow;

// Blocks of an even number of bytes: the words' byte phase alternates with b.
template <int BYTES> struct PfRowEven {
    struct Raw { uint32_t d0, d1, d2; };
    int s, ae, ao, she, sho;
    __device__ __forceinline__ void begin2(int s_, int t, int nib) {   // t: the lane's first byte in block 0
        s = s_;
        ae = t & ~3; she = 8 * (t & 3) + nib;
        t += BYTES;
        ao = t & ~3; sho = 8 * (t & 3) + nib;
    }
    __device__ __forceinline__ Raw load(const uint8_t* l, int b, int) const {
        const uint32_t* w = (const uint32_t*)(l + ((b & 1) ? ao : ae) + 2 * BYTES * (b >> 1));
        return Raw{w[0], w[1], w[2]};
    }
    __device__ __forceinline__ Raw look(const Raw& r, int, const uint32_t*) const { return r; }
    __device__ __forceinline__ uint32_t dw(const uint8_t* l, int b) const { return lds_u16(l, s + BYTES * b); }
};

template <> struct PfRow<T_Q4_0> : PfRowEven<18> {
    typedef Raw Look;
    // elements 8q.. are the low (q < 2) or high nibbles of bytes 8 (q & 1) ..
    __device__ __forceinline__ void begin(const uint8_t*, int s_, int q) {
        begin2(s_, s_ + 2 + 8 * (q & 1), 4 * (q >> 1));
    }
    __device__ __forceinline__ v8h frag(const Raw& r, int b) const {
        const uint32_t sh = (b & 1) ? sho : she;
        return pf_bytes_h(__builtin_amdgcn_alignbit(r.d1, r.d0, sh) & 0x0F0F0F0Fu,
                          __builtin_amdgcn_alignbit(r.d2, r.d1, sh) & 0x0F0F0F0Fu) -
               (_Float16)1032;   // nibble - 8
    }
};

template <> struct PfRow<T_Q8_0> : PfRowEven<34> {
    typedef Raw Look;
    __device__ __forceinline__ void begin(const uint8_t*, int s_, int q) { begin2(s_, s_ + 2 + 8 * q, 0); }
    __device__ __forceinline__ v8h frag(const Raw& r, int b) const {
        const uint32_t sh = (b & 1) ? sho : she;
        return pf_bytes_h(__builtin_amdgcn_alignbit(r.d1, r.d0, sh) ^ 0x80808080u,
                          __builtin_amdgcn_alignbit(r.d2, r.d1, sh) ^ 0x80808080u) -
               (_Float16)1152;   // (byte ^ 0x80) - 128
    }
};

template <> struct PfRow<T_IQ3_S> {
    // superblock [f16 d][qs 64][qh 8][signs 32][scales 4] (gguf_loader.rs:1008-1142):
    // grid entries qs[8b+2q], qs[8b+2q+1] with high bits 2q, 2q+1 of qh[b],
    // signs = byte 4b + q, times 1 + 2 * scale (at most 465: exact in f16)
    struct Raw { uint32_t qs, sg; };
    struct Look { uint2 g0, g1; uint32_t sg; };
    int s;
    uint32_t sc, h0[2], h1[2];   // high bits as 0/1 bytes, byte b & 3 of word b >> 2
    uint32_t d;
    __device__ __forceinline__ void begin(const uint8_t* l, int s_, int q) {
        s = s_;
        d = lds_u16(l, s);
        sc = lds_u32(l, s + 106);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint32_t w = lds_u32(l, s + 66 + 4 * i);
            h0[i] = (w >> (2 * q)) & 0x01010101u;
            h1[i] = (w >> (2 * q + 1)) & 0x01010101u;
        }
    }
    __device__ __forceinline__ Raw load(const uint8_t* l, int b, int q) const {
        return Raw{lds_u16(l, s + 2 + 8 * b + 2 * q), l[s + 74 + 4 * b + q]};
    }
    __device__ __forceinline__ Look look(const Raw& r, int b, const uint32_t* grid) const {
        const uint32_t sel = 0x0C0C0000u | ((uint32_t)(4 + (b & 3)) << 8);
        const uint32_t i0 = __builtin_amdgcn_perm(h0[b >> 2], r.qs, sel);
        const uint32_t i1 = __builtin_amdgcn_perm(h1[b >> 2], r.qs, sel | 1u);
        return Look{*(const uint2*)(grid + 2 * i0), *(const uint2*)(grid + 2 * i1), r.sg};
    }
    __device__ __forceinline__ v8h frag(const Look& k, int b) const {
        // sign bits j and j + 1 to bits 15 and 31: bit j of r is sign j, bit
        // j + 15 too
        const uint32_t r = k.sg | (k.sg << 15);
        const uint4 v = make_uint4(k.g0.x ^ ((r << 15) & 0x80008000u), k.g0.y ^ ((r << 13) & 0x80008000u),
                                   k.g1.x ^ ((r << 11) & 0x80008000u), k.g1.y ^ ((r << 9) & 0x80008000u));
        const _Float16 m = (_Float16)(unsigned short)(((sc >> (4 * b)) & 0xFu) * 2 + 1);
        return __builtin_bit_cast(v8h, v) * m;
    }
    __device__ __forceinline__ uint32_t dw(const uint8_t*, int) const { return d; }
};

// Q4_K / Q5_K: [f16 d][f16 dmin][scales 12]([qh 32])[qs 128] (gguf_loader.rs:1165-1330),
// quant * 6-bit scale (at most 31 * 63 = 1953: exact in f16)
template <int T> struct PfRowK {
    struct Raw { uint32_t d0, d1, d2; };
    typedef Raw Look;
    int s;
    uint32_t w0, s0, s1, s2, h0, h1;   // h0, h1: qh of elements 8q..8q+7, bit b for block b
    __device__ __forceinline__ void begin(const uint8_t* l, int s_, int q) {
        s = s_;
        w0 = lds_u32(l, s);
        s0 = lds_u32(l, s + 4); s1 = lds_u32(l, s + 8); s2 = lds_u32(l, s + 12);
        if constexpr (T == T_Q5_K) { h0 = lds_u32(l, s + 16 + 8 * q); h1 = lds_u32(l, s + 20 + 8 * q); }
    }
    __device__ __forceinline__ Raw load(const uint8_t* l, int b, int q) const {
        constexpr int QS = T == T_Q5_K ? 48 : 16;
        const uint32_t* w = (const uint32_t*)(l + ((s + QS + 8 * q) & ~3) + 32 * (b >> 1));
        return Raw{w[0], w[1], w[2]};
    }
    __device__ __forceinline__ Raw look(const Raw& r, int, const uint32_t*) const { return r; }
    __device__ __forceinline__ v8h frag(const Raw& r, int b) const {
        int sc, m;
        kq_scale_min(s0, s1, s2, b, sc, m);
        const uint32_t sh = 8 * (s & 3) + 4 * (b & 1);
        uint32_t lo = __builtin_amdgcn_alignbit(r.d1, r.d0, sh) & 0x0F0F0F0Fu;
        uint32_t hi = __builtin_amdgcn_alignbit(r.d2, r.d1, sh) & 0x0F0F0F0Fu;
        if constexpr (T == T_Q5_K) {
            lo |= (b < 4 ? h0 << (4 - b) : h0 >> (b - 4)) & 0x10101010u;
            hi |= (b < 4 ? h1 << (4 - b) : h1 >> (b - 4)) & 0x10101010u;
        }
        return (pf_bytes_h(lo, hi) - (_Float16)1024) * (_Float16)(unsigned short)sc;
    }
    __device__ __forceinline__ uint32_t dw(const uint8_t*, int) const { return w0 & 0xFFFFu; }
    __device__ __forceinline__ float neg_dmin() const { return -h2f(w0 >> 16); }
    __device__ __forceinline__ float min_of(int b) const {   // 6-bit min of sub-block b
        int sc, m;
        kq_scale_min(s0, s1, s2, b, sc, m);
        return (float)m;
    }
};
template <> struct PfRow<T_Q4_K> : PfRowK<T_Q4_K> {};
template <> struct PfRow<T_Q5_K> : PfRowK<T_Q5_K> {};

template <> struct PfRow<T_Q6_K> {
    // [ql 128][qh 64][i8 scales 16][f16 d] (gguf_loader.rs:839-917); the two
    // 16-element halves of a block have their own int8 scales, so their
    // products stay apart (frag: q - 32 without a scale)
    struct Raw { uint32_t l0, l1, h0, h1; };
    typedef Raw Look;
    int s;
    uint32_t d;
    __device__ __forceinline__ void begin(const uint8_t* l, int s_, int) {
        s = s_;
        d = lds_u16(l, s + 208);
    }
    __device__ __forceinline__ Raw load(const uint8_t* l, int b, int q) const {
        const int gi = b >> 2, jj = b & 3;
        const int lo = s + 64 * gi + 32 * (jj & 1) + 8 * q, hi = s + 128 + 32 * gi + 8 * q;
        return Raw{lds_u32(l, lo), lds_u32(l, lo + 4), lds_u32(l, hi), lds_u32(l, hi + 4)};
    }
    __device__ __forceinline__ Look look(const Raw& r, int, const uint32_t*) const { return r; }
    __device__ __forceinline__ v8h frag(const Look& r, int b) const {
        const int nsh = 4 * ((b & 3) >> 1), hsh = 2 * (b & 3);
        return pf_bytes_h(((r.l0 >> nsh) & 0x0F0F0F0Fu) | (((r.h0 >> hsh) & 0x03030303u) << 4),
                          ((r.l1 >> nsh) & 0x0F0F0F0Fu) | (((r.h1 >> hsh) & 0x03030303u) << 4)) -
               (_Float16)1056;
    }
    __device__ __forceinline__ uint32_t dw(const uint8_t*, int) const { return d; }
    __device__ __forceinline__ float scale(const uint8_t* l, int b, int half) const {
        return (float)(int)(int8_t)l[s + 192 + 8 * (b >> 2) + 2 * (b & 3) + half];
    }
};

// ---- LDS of one work-group: nw stages (1 or 2) of the weight rows' chunks, two of the
// activation blocks (units of 8 pairs x 2 blocks) and of their scales
// ([pair][block]; K-quants also d_x * sum q_x)
struct PfLds {
    uint8_t* smem;
    uint32_t* sd;
    int wst, xst, dst, nw;   // bytes of a weight and of an activation stage, words of a scale stage
    __device__ __forceinline__ uint8_t* w(int p) const { return smem + p * wst; }
    __device__ __forceinline__ uint8_t* x(int p) const { return smem + nw * wst + p * xst; }
    __device__ __forceinline__ uint32_t* d(int p) const { return sd + p * dst; }
    __device__ __forceinline__ float* s(int p) const { return (float*)(sd + 2 * dst + p * dst); }
};

// One work-group: ns slices of PF_ROWS weight rows (64 at w0, 64 at w1 of the
// first; global row stride rb, slices sstride bytes apart) against 16 * MT pairs, each a row of xh / xd / xs;
// wave w computes the 16-row tiles n = 0, 1 at rows 64 n + 16 w of all pairs:
// acc[n][m][i] = output (pair 16 m + 4 (l / 16) + i, row 64 n + 16 w + l % 16),
// handed to done(slice, acc) while the next slice's first copies are in flight.
// Pair i of np is row list[first + i] when `list` is not null, otherwise row
// first + i; padding rows repeat the last pair.
//
// Weight chunk c + 1 and the activation stage after the current one are
// copied (asynchronously, untracked by the compiler) while the current ones
// are computed.  With chunks of two activation stages, a stage's copies are
// issued before those of a weight chunk, so a wave can wait for the stage
// (vmcnt counts in order) with the weight chunk still in flight: its HBM round
// trip has a whole chunk of work to hide behind.  WDB false: one weight stage
// over the memory of both (shared-expert rows wider than a stage).
template <int T, int MT, int XB, bool WDB, class Done>
__device__ __forceinline__ void pf_gemm(const PfLds& L, const uint8_t* w0, const uint8_t* w1, int64_t rb, int ns,
                                        int64_t sstride, int nbk,
                                        const _Float16* xh, const uint32_t* xd, const float* xs, const int* list,
                                        int first, int np, const uint32_t* grid, Done done) {
    constexpr int NTN = 2, CH = pf_ch<T>(), CB = pf_cb<T>(), SL = pf_sl<T>(), SPC = CH / XB;
    constexpr int NSLOT = pf_row<T>(PF_ROWS) / 16, NWG = (NSLOT + 63) / 64, NIT = (NWG + 3) / 4;
    constexpr int KT = 4 / MT;   // blocks whose scale products one 4-block instruction makes
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nc = nbk / CH;
    float acc[NTN][MT][4];

    int* tok = (int*)L.x(1);   // the rows, a copy per wave (the stage is filled after the first barrier)
    if (list) copy4_lds_untracked(list + first + min(lane, np - 1), tok + 64 * wave);
    // this thread's weight pieces: 16-byte slot `col` of row r, the same every chunk
    const uint8_t* wp[NIT];
    int wcol[NIT];
#pragma unroll
    for (int k = 0; k < NIT; k++) {
        const int cc = (k * 4 + wave) * 64 + lane;
        int r, col;
        if constexpr (pf_skew<T>()) {
            const int g4 = cc / (4 * SL + 1), rem = cc - g4 * (4 * SL + 1);
            r = 4 * g4 + rem / SL;
            col = rem < 4 * SL ? rem % SL : SL;
        } else {
            r = cc / SL;
            col = cc - r * SL;
        }
        wp[k] = (r < 64 ? w0 + (int64_t)r * rb : w1 + (int64_t)(r - 64) * rb) + col * 16;
        wcol[k] = r < PF_ROWS && col < SL ? col * 16 : 1 << 20;
    }
    // weight copy instructions of this wave per chunk (64 consecutive slots
    // hold the first slot of a row, so each has an active lane)
    const int nwi = (NWG - wave + 3) / 4;
    // chunk at byte `off` of the first slice's rows, into stage p
    auto issue_w = [&](int64_t off, int p_) {
        // the span [start & ~15, start + CB) of each row's chunk; an aligned
        // 16-byte piece never leaves the page of the valid bytes it holds
        uint8_t* dst = L.w(WDB ? p_ : 0);
#pragma unroll
        for (int k = 0; k < NIT; k++) {
            const uint8_t* p = wp[k] + off;
            const int pre = (int)((uintptr_t)p & 15);
            if (k * 4 + wave < NWG && wcol[k] < pre + CB) copy16_lds_untracked(p - pre, dst + (k * 4 + wave) * 1024);
        }
    };
    issue_w(0, 0);

    // activation copies: a unit is 8 pairs x 2 blocks (128 contiguous bytes of
    // a pair's row per 8 lanes: whole cache lines); a stage has 2 * MT groups
    // of 8 pairs x XB / 2 pairs of blocks
    constexpr int NXP = MT > 1 ? MT / 2 : 1, NXB = MT > 1 ? XB / 2 : XB / 4;
    const int64_t nb = nbk;
    if (list) wait_vm_n(nwi);   // the rows, with the first weight chunk in flight
    auto rowof = [&](int i) { return list ? tok[64 * wave + i] : first + min(i, np - 1); };
    const uint8_t* xp[NXP];
#pragma unroll
    for (int j = 0; j < NXP; j++) {
        const int grp = MT > 1 ? wave + 4 * j : wave & 1, r = lane >> 3;
        xp[j] = (const uint8_t*)(xh + (int64_t)rowof(8 * grp + r) * (nb * 32)) + (MT > 1 ? 0 : 128 * NXB * (wave >> 1)) +
                16 * ((lane & 7) ^ r);
    }
    // scales (wave 0), K-quants' d_x * sum q_x (wave 1): a pair's 4 blocks per lane
    const uint32_t* dp = (wave ? (const uint32_t*)xs : xd) + (lane < 16 * MT ? (int64_t)rowof(lane) * nb : 0);

    auto issue_x = [&](int st, int p) {   // activation stage st of the row, into stage p
#pragma unroll
        for (int j = 0; j < NXP; j++)
#pragma unroll
            for (int k = 0; k < NXB; k++) {
                const int unit = MT > 1 ? XB / 2 * (wave + 4 * j) + k : XB / 2 * (wave & 1) + NXB * (wave >> 1) + k;
                copy16_lds_untracked(xp[j] + (int64_t)st * (64 * XB) + 128 * k, L.x(p) + unit * 1024);
            }
        if (wave < (pf_kq<T>() ? 2 : 1) && lane < 16 * MT)
#pragma unroll
            for (int k = 0; k < XB / 4; k++)   // [quad of blocks][pair][4]
                copy16_lds_untracked(dp + st * XB + 4 * k, (wave ? (uint32_t*)L.s(p) : L.d(p)) + 64 * MT * k);
    };
    // the lane's rows: low address bits, for the chunk's start in its LDS row
    int rlow[NTN], rlds[NTN];
#pragma unroll
    for (int n = 0; n < NTN; n++) {
        rlow[n] = (int)((uintptr_t)(n ? w1 : w0) + (uintptr_t)((16 * wave + c) * rb)) & 15;
        rlds[n] = pf_row<T>(64 * n + 16 * wave + c);
    }
    // the lane's place in an activation stage (elements 8q.. of pair c of a
    // tile; the 16-byte pieces of a pair's 128 bytes are permuted by the pair
    // so that 8 lanes read 8 distinct places modulo 128 bytes) and among the
    // scales (block q / MT of pair c of tile q % MT)
    const int xo = (c >> 3) * (512 * XB) + (c & 7) * 128 + (q ^ (c & 7)) * 16;
    const int dxo = (16 * (q % MT) + c) * 4 + q / MT;

    issue_x(0, 0);
    int v = 0;             // chunks done; weight stage v & 1, activation stages (SPC * v + ...) & 1
    int64_t woff = 0;      // byte offset of the chunk in the first slice's rows
    for (int sl = 0; sl < ns; sl++) {
#pragma unroll
        for (int n = 0; n < NTN; n++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int i = 0; i < 4; i++) acc[n][m][i] = 0.0f;
        for (int ch = 0; ch < nc; ch++) {
            const bool last = ch + 1 == nc && sl + 1 == ns;
            // the next chunk, and its (first) activation stage
            const int64_t wnext = ch + 1 < nc ? woff + CB : (int64_t)(sl + 1) * sstride;
            const int xnext = ch + 1 < nc ? SPC * (ch + 1) : 0;
            // A chunk's (block, row tile) groups in one straight line.  While the
            // matrix cores run group g, the vector ALU rescales group g - 1,
            // finishes the weights of g + 1 and starts the lookups of g + 2, whose
            // LDS reads were issued one group before: no step waits on the one
            // right before it.  (Left to itself the compiler moves each product
            // next to its use.)
            constexpr int NG = CH * NTN, HG = XB * NTN;
            typedef typename PfRow<T>::Raw Raw;
            typedef typename PfRow<T>::Look Look;
            const uint8_t* wl = L.w(WDB ? v & 1 : 0);
            PfRow<T> row[NTN];
            Raw raw[NG];
            Look look[NG];
            v8h w[NG], a[CH][MT];
            v4f s0[NG][MT], s1[NG][MT];
            v16f t[NG];
            uint32_t dx[CH], dwv[NG];
            float m0[NG], m1[NG], ks[CH][MT][4];   // Q6_K half scales; K-quants: d_x * sum q_x of the lane's outputs
            const v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
            const v16f z16 = {0.0f};
            auto do_load = [&](int g) {
                const int n = g % NTN, b = g / NTN;
                raw[g] = row[n].load(wl, b, q);
                if (b % KT == 0) dwv[g] = row[n].dw(wl, b + q / MT);   // lane group q: block b + q / MT, pair tile q % MT
                if constexpr (T == T_Q6_K) { m0[g] = row[n].scale(wl, b, 0); m1[g] = row[n].scale(wl, b, 1); }
            };
            auto do_look = [&](int g) { look[g] = row[g % NTN].look(raw[g], g / NTN, grid); };
            auto do_frag = [&](int g) { w[g] = row[g % NTN].frag(look[g], g / NTN); };
            auto do_a = [&](int b) {
                const int st = SPC * v + b / XB, bb = b % XB, dq = 64 * MT * (bb >> 2) + (bb & 3);
#pragma unroll
                for (int m = 0; m < MT; m++)
                    a[b][m] = *(const v8h*)(L.x(st & 1) + m * (1024 * XB) + (bb >> 1) * 1024 + (bb & 1 ? xo ^ 64 : xo));
                if (b % KT == 0) dx[b] = L.d(st & 1)[dq + dxo];
                if constexpr (pf_kq<T>()) {
#pragma unroll
                    for (int m = 0; m < MT; m++)
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            ks[b][m][i] = L.s(st & 1)[(16 * m + 4 * q + i) * 4 + dq];
                        }
                }
            };
            auto do_mma = [&](int g) {
                const int b = g / NTN;
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    if constexpr (T == T_Q6_K) {
                        const v8h zero = {};
                        s0[g][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[b][m], q < 2 ? w[g] : zero, z, 0, 0, 0);
                        s1[g][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[b][m], q < 2 ? zero : w[g], z, 0, 0, 0);
                    } else {
                        s0[g][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[b][m], w[g], z, 0, 0, 0);
                    }
                }
                if (b % KT == 0) {
                    // scale products of KT blocks x MT pair tiles
                    auto h4 = [](uint32_t h) { return __builtin_bit_cast(v4h, make_uint2(h, 0)); };
                    t[g] = __builtin_amdgcn_mfma_f32_16x16x4f16(h4(dx[b]), h4(dwv[g]), z16, 0, 0, 0);
                }
            };
            auto do_acc = [&](int g) {
                const int n = g % NTN, b = g / NTN, tg = (b - b % KT) * NTN + n;   // the group that made the scales
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int ti = 4 * (m + MT * (b % KT)) + i;
                        // Q6_K: lo * sc0 + hi * sc1, both products and the sum exact
                        const float sv = T == T_Q6_K ? __builtin_fmaf(s1[g][m][i], m1[g], s0[g][m][i] * m0[g]) : s0[g][m][i];
                        float o = __builtin_fmaf(t[tg][ti], sv, acc[n][m][i]);
                        // the K-quants' min term fmaf(-(f32(dmin) * f32(d_x)), (float)(m * sum q_x),
                        // acc), its exact product as -(dmin * m) times d_x * sum q_x (both exact)
                        if constexpr (pf_kq<T>()) o = __builtin_fmaf(row[n].neg_dmin() * row[n].min_of(b), ks[b][m][i], o);
                        asm volatile("" : "+v"(o));   // the rescale stays in its group (it would sink below the products)
                        acc[n][m][i] = o;
                    }
            };
            wait_vm<0>();
            lds_barrier();   // weight chunk ch and its (first) activation stage landed: every wave's share
            if (SPC > 1) issue_x(SPC * ch + 1, (SPC * v + 1) & 1);
            else if (!last) issue_x(xnext, (v + 1) & 1);
            if (WDB && !last) issue_w(wnext, (v + 1) & 1);
#pragma unroll
            for (int n = 0; n < NTN; n++) row[n].begin(wl, rlds[n] + ((rlow[n] + (int)woff) & 15), q);
            do_load(0);
            do_load(1);
            do_load(2);
            do_a(0);
            do_look(0);
            do_look(1);
            do_frag(0);
#pragma unroll
            for (int g = 0; g < NG; g++) {
                if (SPC > 1 && g == HG) {
                    // the second activation stage landed; the next weight chunk stays in flight
                    if (WDB && !last) wait_vm_n(nwi);
                    else wait_vm<0>();
                    lds_barrier();
                    if (!last) issue_x(xnext, (SPC * v + 2) & 1);
                    do_a(XB);
                }
                if (g + 3 < NG) do_load(g + 3);
                if (g % NTN == NTN - 1 && g + 1 != HG && g + 1 < NG) do_a(g / NTN + 1);
                if (g + 2 < NG) do_look(g + 2);
                do_mma(g);
                if (g > 0) do_acc(g - 1);
                if (g + 1 < NG) do_frag(g + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            do_acc(NG - 1);
            if (!WDB && !last) {
                lds_barrier();   // every wave is done with the chunk
                issue_w(wnext, 0);
            }
            v++;
            woff = wnext;
        }
        done(sl, acc);
    }
}

// ---- the two expert launches

// One weight stage at 32 pairs per tile: then a third work-group fits the CU,
// which hides a chunk's copies better than a second stage (512 tokens Q4_0
// gate/up 110 -> 104 us, down 61 -> 55; IQ3_S + Q5_K gate/up 128 -> 117).  16
// pairs have three work-groups with two stages (one: 45 tokens IQ3_S + Q5_K
// 76 -> 82 us), but two where the types are IQ3_S and Q4_0 / Q8_0 (the wider stage
// of the one and the codebook of the other: 54,816 bytes); 64 pairs two either
// way, by their registers.  Not for the down
// launch next to a shared type of two-part blocks: its loop holds up to 199
// registers, and in a third of the register file Q4_K / Q5_K / Q6_K spilled 25 /
// 34 / 36 of them (512 tokens, one stage / two: Q4_0 + Q6_K 219 / 203 us, Q4_0 +
// Q5_K 213 / 201, IQ3_S + Q6_K 227 / 218, IQ3_S + Q5_K 224 / 216, IQ3_S + Q4_K
// 220 / 216; 16 pairs at a time in one stage are 1-2 % faster still with IQ3_S
// experts but 17 % slower for 256 tokens at H = F = 1024).  The gate/up launch
// (at most 7 spilled) keeps one: with two, IQ3_S + Q6_K 220 us, + Q5_K 221, + Q4_K 221.
template <int TS, int MT, bool DOWN>
constexpr bool pf_single() { return MT == 2 && !(DOWN && (pf_kq<TS>() || TS == T_Q6_K)); }
// bytes of a weight stage next to experts of type TE: a shared type of at most
// 10 slots per row has two stages too, a wider one (and the K-quants) a single
// stage over both; with one weight stage it holds either
template <int TE, int TS, bool ONE>
constexpr int pf_wst2() {
    return pf_wst<TS>() > pf_wst<TE>() && (ONE || (pf_sl<TS>() <= 10 && !pf_kq<TS>())) ? pf_wst<TS>() : pf_wst<TE>();
}
template <int T, int TE, int TS, bool ONE>
constexpr bool pf_wdb() { return !ONE && pf_wst<T>() <= pf_wst2<TE, TS, ONE>(); }
// Blocks of the activation rows per LDS stage, M tiles of 16 pairs at a time:
// a whole chunk (one barrier less) where two weight stages leave two
// work-groups per CU either way: in the tiles of up to 32 pairs of the 64-pair
// kernels, and in the 32-pair kernels of two weight stages (with four blocks, 800 tokens: IQ3_S + Q6_K 268 -> 274 us,
// IQ3_S + Q8_0 254 -> 258, Q4_0 235 -> 238)
template <int T, int M, bool ONE>
constexpr int pf_xb() { return pf_ch<T>() == 8 && M == 2 && !ONE ? 8 : 4; }
// blocks x 16-pair tiles of an activation stage
template <int MT, bool ONE>
constexpr int pf_xu() { return MT == 2 && !ONE ? 16 : 4 * MT; }

// Work-group -> (tile, slice of rows); pairs 0: none.  The hardware deals
// work-groups to the 8 XCDs round-robin, and the slices of one tile follow each
// other on one XCD: its activation rows are fetched into that L2 once, and
// the tiles of one expert (consecutive) share its weights there.  The shared
// expert's tiles (full ones, and of the slower types) are dealt apart from the
// experts' and come first: with them at the end of one list a single XCD had
// them all, 4096 tokens IQ3_S + Q5_K gate/up 774 against 562 us.
//  * whole tiles: entry 8 g + x is XCD x's g-th, the shared expert's dealt one
//    by one, the experts' in contiguous eighths, pairs 0 in unused entries;
//  * otherwise XCD x has a contiguous eighth of each part's (tile, slice) list:
//    entry 0 has the number of the experts' tiles, then follow the shared
//    expert's and the experts'.  Few tiles are bound by each XCD's weight
//    stream, and by whole tiles an XCD had up to two more than another (35
//    tiles: 6 and none; halves of tiles: still 13 % more than the average).
// Whole tiles / slices (us): 12 tokens, H = 4096, F = 1024, 64 experts, top-4
// Q8_0 144 / 112, IQ3_S + Q5_K 117 / 95; H = 2048, F = 512, 256 experts, top-8:
// 9 tokens Q8_0 77 / 64, IQ3_S + Q5_K 72 / 62.  Many tiles are even enough whole,
// without the load of the count that the tile's waits for (PF_WHOLE_TILES).
__host__ __device__ constexpr int pf_eighth(int n) { return (n + 7) >> 3; }
__device__ __forceinline__ int4 pf_place(const PfArgs& a, int nslice, int& sl) {   // nslice: work-groups per tile
    const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
    if (a.whole) {
        const int g = k / nslice;
        sl = k - g * nslice;
        return a.tiles[8 * g + x];
    }
    const int ps = pf_eighth(a.nsh * nslice);
    const bool sh = k < ps;
    const int n = (sh ? a.nsh : a.tiles[0].x) * nslice, per = pf_eighth(n), i = sh ? k : k - ps;
    const int w = x * per + i, t = w / nslice;
    sl = w - t * nslice;
    if (i >= per || w >= n) return make_int4(0, 0, 0, 0);
    return a.tiles[1 + (sh ? 0 : a.nsh) + t];
}
// work-groups of a launch
inline int pf_grid(const PfArgs& a, int nslice) {
    if (a.whole) return 8 * (pf_eighth(a.nsh) + pf_eighth(a.max_tiles)) * nslice;
    return 8 * (pf_eighth(a.nsh * nslice) + pf_eighth(a.max_tiles * nslice));
}

// LDS arrays of a work-group
#define PF_LDS_ARRAYS                                                                                       \
    constexpr bool IQ = TE == T_IQ3_S || TS == T_IQ3_S, KQ = pf_kq<TS>();                                   \
    constexpr int NW = ONE ? 1 : 2, XU = pf_xu<MT, ONE>(), WST = pf_wst2<TE, TS, ONE>();                     \
    __shared__ __attribute__((aligned(16))) uint8_t smem[NW * WST + 2 * XU * 1024];                         \
    __shared__ __attribute__((aligned(16))) uint32_t sd[(KQ ? 4 : 2) * XU * 16];                            \
    __shared__ __attribute__((aligned(16))) uint32_t grid[IQ ? 1024 : 1];                                   \
    const PfLds L{smem, sd, WST, XU * 1024, XU * 16, NW};                                                   \
    /* the codebook, one kilobyte per wave; landed with the first weight chunk */                           \
    if constexpr (IQ)                                                                                       \
        copy16_lds_untracked((const uint4*)c_iq3s_hgrid.w + threadIdx.x, (uint4*)grid + (threadIdx.x & ~63u))

// The tile's pairs against type T: run(type, pair tiles, first position, pairs)
template <int TE, int TS, int MT, int MKQ, class Run>
__device__ __forceinline__ void pf_dispatch(const int4& ti, bool sh, Run run) {
    auto with = [&](auto ttag) {
        // Q6_K's second products leave registers for 32 pairs at a time, the
        // K-quants' min terms for 16 * MKQ
        constexpr int T = decltype(ttag)::value, MX = T == T_Q6_K ? 2 : pf_kq<T>() ? MKQ : 4,
                      M = MT < MX ? MT : MX;
        if constexpr (M < MT) {
            for (int p = 0; p < ti.z; p += PF_PT * M) {
                run(ttag, std::integral_constant<int, M>{}, ti.y + p, min(ti.z - p, PF_PT * M));
                lds_barrier();   // every wave is done with the stages
            }
        } else if (MT > 1 && ti.z <= PF_PT * MT / 2) {
            run(ttag, std::integral_constant<int, (MT > 1 ? MT / 2 : 1)>{}, ti.y, ti.z);
        } else {
            run(ttag, std::integral_constant<int, MT>{}, ti.y, ti.z);
        }
    };
    if (TE == TS || !sh) with(std::integral_constant<int, TE>{});
    else if constexpr (TE != TS) with(std::integral_constant<int, TS>{});
}

// P4: F / 64 work-groups per tile (pf_place): h = silu(gate) * up of 64 rows of
// F for a tile's pairs, as Q8_1 blocks (by position in spairs).  (Two and four
// slices of rows per work-group, the next one's copies in flight during this
// epilogue, measured slower: 512 tokens Q4_0 108 -> 118 and 144 us -- fewer
// work-groups, and the loop's state held across the epilogue.)
template <int TE, int TS, int MT>
__global__ __launch_bounds__(PF_THREADS, (pf_single<TS, MT, false>() ? 3 : 2)) void k_pf_gate_up(PfArgs a) {
    constexpr bool ONE = pf_single<TS, MT, false>();
    int sl;
    const int4 ti = pf_place(a, a.F / 64, sl);
    if (ti.z == 0) return;
    PF_LDS_ARRAYS;
    float* ex = (float*)sd;
    const int e = ti.x, f0 = sl * 64;
    const bool sh = e == a.E;
    const uint8_t* g = sh ? a.sh_gate : a.gate + (int64_t)e * a.sg;
    const uint8_t* u = sh ? a.sh_up : a.up + (int64_t)e * a.su;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, c = lane & 15;
    pf_dispatch<TE, TS, MT, 4>(ti, sh, [&](auto ttag, auto mtag, int start, int np) {
        constexpr int T = decltype(ttag)::value, M = decltype(mtag)::value;
        const int64_t rb = row_bytes(T, a.H);
        pf_gemm<T, M, pf_xb<T, M, ONE>(), pf_wdb<T, TE, TS, ONE>()>(L, g + f0 * rb, u + f0 * rb, rb, 1, 64 * rb, a.H / QK, a.xh, a.xd,
                                           a.xs, a.stok, start, np, grid, [&](int, float (&acc)[2][M][4]) {
            // wave w has gate and up of rows f0 + 16 w + c: half a block of h.
            // Q8_1 as k_quantize_q8_1: the halves' maxima (K-quants: quant
            // sums) are exchanged through LDS (the scale stages, free now)
            lds_barrier();   // every wave is done with them
            float am[M][4];
#pragma unroll
            for (int m = 0; m < M; m++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float h = det_silu(acc[0][m][i]) * acc[1][m][i];
                    acc[0][m][i] = h;
                    float v = __builtin_fabsf(h);
                    v = __builtin_fmaxf(v, xlane<8>(v));
                    v = __builtin_fmaxf(v, xlane<4>(v));
                    v = __builtin_fmaxf(v, xlane<2>(v));
                    am[m][i] = __builtin_fmaxf(v, xlane<1>(v));
                }
                if (c == 0)
                    *(float4*)(ex + wave * 16 * M + 16 * m + 4 * q) = make_float4(am[m][0], am[m][1], am[m][2], am[m][3]);
            }
            lds_barrier();
            const int64_t nb = a.F / QK;
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float4 o = *(const float4*)(ex + (wave ^ 1) * 16 * M + 16 * m + 4 * q);
                const float ov[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int p = 16 * m + 4 * q + i;
                    const float amax = __builtin_fmaxf(am[m][i], ov[i]), d = amax / 127.0f;
                    // (int8_t): where d underflows to 0 the byte the Q8_1 block would hold
                    const int qv = amax == 0.0f ? 0 : (int8_t)(int)__builtin_roundf(acc[0][m][i] / d);
                    acc[1][m][i] = (float)qv;
                    am[m][i] = h2f(f2h(d));
                    if (p < np) {
                        a.hh[(int64_t)(start + p) * a.F + f0 + 16 * wave + c] = (_Float16)qv;
                        if (c == 0 && (wave & 1) == 0) a.hd[(start + p) * nb + (f0 >> 5) + (wave >> 1)] = f2h(d);
                    }
                }
            }
            if constexpr (pf_kq<T>()) {
                lds_barrier();
#pragma unroll
                for (int m = 0; m < M; m++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float v = slot_reduce16(acc[1][m][i]);   // exact: integers below 2^12
                        acc[1][m][i] = v;
                        if (c == 0) ex[wave * 16 * M + 16 * m + 4 * q + i] = v;
                    }
                lds_barrier();
#pragma unroll
                for (int m = 0; m < M; m++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int p = 16 * m + 4 * q + i;
                        if (c == 0 && (wave & 1) == 0 && p < np)
                            a.hs[(start + p) * nb + (f0 >> 5) + (wave >> 1)] = am[m][i] * (acc[1][m][i] + ex[(wave ^ 1) * 16 * M + p]);
                    }
            }
        });
    });
}

// P5: H / (128 dn_ns) work-groups per tile (pf_place): slices of 128 down rows
// of a tile's pairs, K = F, by pair id.  K is short (16 blocks at F = 512), so
// a work-group of a large launch takes two slices and starts the second's copies
// before it stores the first's outputs: 4096 tokens IQ3_S 248 -> 241 us, 1777
// tokens Q8_0 130 -> 121 us.
template <int TE, int TS, int MT>
__global__ __launch_bounds__(PF_THREADS, (pf_single<TS, MT, true>() ? 3 : 2)) void k_pf_down(PfArgs a) {
    constexpr bool ONE = pf_single<TS, MT, true>();
    int sl;
    const int4 ti = pf_place(a, a.H / (PF_ROWS * a.dn_ns), sl);
    if (ti.z == 0) return;
    PF_LDS_ARRAYS;
    const int e = ti.x, r0 = sl * a.dn_ns * PF_ROWS;
    const bool sh = e == a.E;
    const uint8_t* d = sh ? a.sh_down : a.down + (int64_t)e * a.sd;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, c = lane & 15;
    pf_dispatch<TE, TS, MT, 2>(ti, sh, [&](auto ttag, auto mtag, int start, int np) {
        constexpr int T = decltype(ttag)::value, M = decltype(mtag)::value;
        const int64_t rb = row_bytes(T, a.F);
        int prs[M][4];   // read here: a load between the slices would wait for the copies in flight
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) prs[m][i] = a.spairs[start + min(16 * m + 4 * q + i, np - 1)];
        pf_gemm<T, M, pf_xb<T, M, ONE>(), pf_wdb<T, TE, TS, ONE>()>(L, d + r0 * rb, d + (r0 + 64) * rb, rb, a.dn_ns, PF_ROWS * rb, a.F / QK,
                                           a.hh, a.hd, a.hs, nullptr, start, np, grid, [&](int s, float (&acc)[2][M][4]) {
            const int r = r0 + s * PF_ROWS + 16 * wave + c;
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (16 * m + 4 * q + i < np) {
                        float* o = a.dn + (int64_t)prs[m][i] * a.H + r;
                        o[0] = acc[0][m][i];
                        o[64] = acc[1][m][i];
                    }
        });
    });
}

template <int TE, int TS, int MT>
void pf_launch_mt(const PfArgs& a, hipStream_t s) {
    hipLaunchKernelGGL((k_pf_gate_up<TE, TS, MT>), dim3(pf_grid(a, a.F / 64)), dim3(PF_THREADS), 0, s, a);
    hipLaunchKernelGGL((k_pf_down<TE, TS, MT>), dim3(pf_grid(a, a.H / (PF_ROWS * a.dn_ns))), dim3(PF_THREADS), 0, s, a);
}

// gate/up and down launches of one expert type, a.tile_pairs = 16 * MT pairs per tile
template <int TE>
void pf_launch_experts(const PfArgs& a, int ts, hipStream_t s) {
    auto go = [&](auto tag) {
        constexpr int TS = decltype(tag)::value;
        if (a.tile_pairs == PF_PT) pf_launch_mt<TE, TS, 1>(a, s);
        else if (a.tile_pairs == 2 * PF_PT) pf_launch_mt<TE, TS, 2>(a, s);
        else pf_launch_mt<TE, TS, 4>(a, s);
    };
    if (ts == T_Q4_0) go(std::integral_constant<int, T_Q4_0>{});
    else if (ts == T_Q8_0) go(std::integral_constant<int, T_Q8_0>{});
    else if (ts == T_Q4_K) go(std::integral_constant<int, T_Q4_K>{});
    else if (ts == T_Q5_K) go(std::integral_constant<int, T_Q5_K>{});
    else if (ts == T_Q6_K) go(std::integral_constant<int, T_Q6_K>{});
    else go(std::integral_constant<int, T_IQ3_S>{});
}
extern template void pf_launch_experts<T_Q4_0>(const PfArgs&, int, hipStream_t);
extern template void pf_launch_experts<T_Q8_0>(const PfArgs&, int, hipStream_t);
extern template void pf_launch_experts<T_IQ3_S>(const PfArgs&, int, hipStream_t);

}  // namespace chimere
