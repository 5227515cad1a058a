// mmvq.hip -- block-quantized GEMV (Q8_0 / Q4_0 / IQ3_S / Q4_K / Q5_K / Q6_K /
// MXFP4 weights x Q8_1 activations) for 1..8 tokens, plain /
// batched-by-expert-id / debug dots.
//
// Work-group = 256 threads = 16 row groups of 16 lanes; one tile = 16
// consecutive rows, streamed through LDS by tile_gemv (which documents the
// fp32 order: L=16 lanes per row, G=1).
#include "api_internal.h"
#include "common.h"
#include "tile_gemv.h"

namespace chimere {

void launch_quantize_q8_1(const float* x, void* out, int64_t ncols, int64_t ncols_padded,
                          int64_t nrows, hipStream_t s);

extern __constant__ uint32_t c_iq3s_grid_mmvq[512];
__constant__ uint32_t c_iq3s_grid_mmvq[512] = CHIMERE_IQ3S_GRID_INIT;

struct MmvqArgs {
    const uint8_t* W;
    const uint8_t* x;
    float* y;
    int ncols, nrows, ntok;
    int64_t x_tok_stride;   // bytes between tokens' Q8_1 rows
    int64_t y_tok_stride;   // floats between tokens' outputs
    const int* ids;         // slot k -> expert ids[k]; NULL: expert k
    int64_t w_slot_stride;  // bytes per expert
    int64_t x_slot_stride;  // bytes between slots' inputs (0: shared)
    int64_t y_slot_stride;  // floats between slots' outputs
    // f32 entry points, one launch: x is the f32 row; the first work-group
    // leaves its Q8_1 blocks, zero blocks up to raw_blocks, in raw
    uint8_t* raw;
    int raw_blocks;
};

// The zero blocks past the row's own in the caller's Q8_1 scratch
__device__ __forceinline__ void raw_padding(const MmvqArgs& a) {
    uint32_t* o = (uint32_t*)a.raw;
    for (int i = a.ncols / QK * (Q8_1_BYTES / 4) + threadIdx.x; i < a.raw_blocks * (Q8_1_BYTES / 4); i += GEMV_THREADS)
        o[i] = 0;
}

// Blocks per K chunk of the GEMV tile: 64 for every type, which puts a
// 2048-column Q8_0 row in one chunk (one exposed round trip per work-group
// instead of two: 4096 x 2048 5.45 -> 4.75 us).  Larger chunks for the
// K-quants / MXFP4 (a 4096-column row in one) and the double-buffered tile
// with 32- or 64-block chunks were measured slower: fewer work-groups fit a
// CU, and at 64 blocks four are resident per CU already.
constexpr int MMVQ_BLOCKS = 64;

// LDS row padding of the tile (bytes): with it the 4 rows a wave reads at
// once start on different banks (from a model of the block reads' bank
// conflicts: Q4_0 1152 -> 1200 B, Q8_0 2176 -> 2224 B, IQ3_S 880 -> 960 B)
template <int T>
constexpr int mmvq_pad() { return T == T_Q4_0 || T == T_Q4_0S || T == T_Q8_0 ? 48 : (T == T_IQ3_S ? 80 : 0); }

// bytes of the GEMV tile: padded rows, or 16-byte spans of unaligned ones
template <int T>
constexpr int mmvq_tile() {
    constexpr int CB = chunk_bytes<T>(MMVQ_BLOCKS), P = mmvq_pad<T>(), S = stage_dw<T>() ? ((CB + 30) & ~15) - CB : 0;
    return TILE_ROWS * (CB + (P > S ? P : S)) + 16;
}

// XF32: the f32 entry points' row, quantized by every work-group for itself
template <int T, int NTOK, bool XF32 = false>
__global__ __launch_bounds__(GEMV_THREADS) void k_mmvq(MmvqArgs a) {
    constexpr int CBLK = MMVQ_BLOCKS;
    constexpr int PAD = mmvq_pad<T>();
    __shared__ __attribute__((aligned(16))) uint8_t tile[mmvq_tile<T>()];
    __shared__ XLds xs[NTOK][CBLK];
    __shared__ uint32_t grid[T == T_IQ3_S ? 512 : 1];

    const int tid = threadIdx.x;
    const int g = tid >> 4, j = tid & 15;
    const int slot = blockIdx.y;
    const int r0 = blockIdx.x * TILE_ROWS;
    const int nr = min(TILE_ROWS, a.nrows - r0);
    const int64_t e = a.ids ? (int64_t)a.ids[slot] : (int64_t)slot;
    const int64_t rb = row_bytes(T == T_Q4_0S ? T_Q4_0 : T, a.ncols);
    if constexpr (T == T_IQ3_S)
        for (int i = tid; i < 512; i += GEMV_THREADS) grid[i] = c_iq3s_grid_mmvq[i];

    uint8_t* raw = nullptr;
    if (XF32 && blockIdx.x == 0) {
        raw = a.raw;
        raw_padding(a);
    }
    float acc[1][NTOK];
    tile_gemv<T, NTOK, TILE_ROWS, 1, CBLK, CPOL_STREAM, PAD, true, XF32>(tile, &xs[0][0], grid,
                                     a.W + e * a.w_slot_stride + (int64_t)r0 * rb, nr,
                                     nullptr, 0, rb, a.ncols, a.x + slot * a.x_slot_stride, a.x_tok_stride,
                                     nullptr, a.ntok, acc, raw);
    if (g < nr) {
#pragma unroll
        for (int t = 0; t < NTOK; t++) {
            if (t < a.ntok) {
                const float v = slot_reduce16(acc[0][t]);
                if (j == 0) a.y[slot * a.y_slot_stride + t * a.y_tok_stride + r0 + g] = v;
            }
        }
    }
}

// Several tokens: the block dots on v_mfma_i32_4x4x4_16b_i8, whose 16
// independent 4x4 products are the 16 slots of the fp32 order: lane 4 j + i
// decodes block j (mod 16) of row i of its wave's four rows and is the B column
// of token 4 n + i, so a wave makes the exact int32 dots of 4 rows x 4 tokens x
// 16 blocks in eight instructions, and acc[n][r] of lane 4 j + i is slot j of
// (row r, token 4 n + i).  With the dots as eight v_dot4 per (block, token),
// every lane read every token's block from LDS: 151936x2048 Q6_K, 8 tokens, was
// bound by those reads (320 bytes per lane and block) and its vector ALU (about
// 200 instructions per lane and block): 106 -> 83 us.  The tokens' blocks stay
// raw in LDS: decoded there by every work-group (512 blocks for its 16 rows) the
// same case took 89 us, Q4_0 78 us against 58.
// LDS bytes between tokens' rows of a chunk (raw Q8_1 blocks, copied
// asynchronously): 16 more than the blocks', so that the four tokens a lane
// quad reads are on different banks
constexpr int XTOK_ROW = MMVQ_BLOCKS * Q8_1_BYTES + 16;
typedef int v4i __attribute__((ext_vector_type(4)));

// value of lane 4 j + R of the quad
template <int R>
__device__ __forceinline__ float quad_of(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x55 * R, 0xF, 0xF, true));
}

template <int T, int NG>
__global__ __launch_bounds__(GEMV_THREADS) void k_mmvq_tok(MmvqArgs a) {
    constexpr int CBLK = MMVQ_BLOCKS, CB = chunk_bytes<T>(CBLK), PAD = mmvq_pad<T>();
    __shared__ __attribute__((aligned(16))) uint8_t tile[mmvq_tile<T>()];
    __shared__ __attribute__((aligned(16))) uint8_t xs[4 * NG * XTOK_ROW];
    __shared__ uint32_t grid[T == T_IQ3_S ? 512 : 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane >> 2, i = lane & 3;
    const int r0 = blockIdx.x * TILE_ROWS, nr = min(TILE_ROWS, a.nrows - r0);
    const int64_t rb = row_bytes(T, a.ncols);
    const uint8_t* W = a.W + (int64_t)r0 * rb;
    const int nb = a.ncols / QK;
    if constexpr (T == T_IQ3_S)
        for (int k = tid; k < 512; k += GEMV_THREADS) grid[k] = c_iq3s_grid_mmvq[k];
    float acc[NG][4];
#pragma unroll
    for (int n = 0; n < NG; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[n][r] = 0.0f;
    for (int b0 = 0; b0 < nb; b0 += CBLK) {
        const int cb = min(CBLK, nb - b0), seg = chunk_bytes<T>(cb);
        const int64_t goff = (int64_t)b0 / (QTraits<T>::ELEMS / QK) * QTraits<T>::BYTES;
        const bool al16 = (((uintptr_t)W | (uintptr_t)rb | (uintptr_t)goff | (uintptr_t)seg) & 15) == 0;
        const bool xal = (((uintptr_t)a.x | (uintptr_t)a.x_tok_stride | (uintptr_t)(cb * Q8_1_BYTES)) & 15) == 0;
        const bool spans = span_rows<T>(W + goff, rb, nr, seg);
        const int lseg = spans ? span_stride(seg) : PAD && al16 ? seg + PAD : seg;
        __syncthreads();   // every wave is done with the previous chunk
        bool staged = false;
        if constexpr (CB % 16 == 0)
            if (al16 && cb == CBLK) {
                stage_rows_fixed<CB, CB + PAD, 16, TILE_ROWS, GEMV_THREADS, CPOL_STREAM, true>(tile, W + goff, nr, nullptr,
                                                                                             rb, nr, tid);
                staged = true;
            }
        if (spans) stage_row_spans<CPOL_STREAM>(tile, W + goff, rb, nr, seg, tid, GEMV_THREADS);
        else if (!staged) stage_rows<stage_dw<T>(), CPOL_STREAM>(tile, W + goff, rb, nr, seg, tid, GEMV_THREADS, lseg);
        // tokens past the last repeat it (their sums are not stored); a
        // wave copies whole tokens
#pragma unroll
        for (int k = 0; k < NG; k++) {
            const int t = 4 * k + wave;
            const uint8_t* src = a.x + min(t, a.ntok - 1) * a.x_tok_stride + (int64_t)b0 * Q8_1_BYTES;
            if (xal)
                for (int c = 0; c < cb * Q8_1_BYTES / 16; c += 64) {
                    if (c + lane < cb * Q8_1_BYTES / 16)
                        __builtin_amdgcn_global_load_lds((const glb_void_t*)(src + (c + lane) * 16),
                                                         (lds_void_t*)(xs + t * XTOK_ROW + c * 16), 16, 0, 0);
                }
            else
                for (int c = 0; c < cb * Q8_1_BYTES / 4; c += 64)
                    if (c + lane < cb * Q8_1_BYTES / 4)
                        __builtin_amdgcn_global_load_lds((const glb_void_t*)(src + (c + lane) * 4),
                                                         (lds_void_t*)(xs + t * XTOK_ROW + c * 4), 4, 0, 0);
        }
        lds_copy_wait();
        __syncthreads();
        const int ri = min(4 * wave + i, nr - 1);   // rows past the last repeat it
        const uint8_t* row = tile + ri * lseg;
        const int pre = spans ? (int)((uintptr_t)(W + goff + ri * rb) & 15) : 0;
#pragma unroll 1
        for (int bg = 0; bg < cb; bg += SLOTS) {
            const bool in = bg + j < cb;
            const int b = in ? bg + j : cb - 1;
            WBlk w;
            block_decode<T>(row, b, grid, w, pre);
            const float mu = T == T_IQ3_S || T == T_Q4_K || T == T_Q5_K || T == T_Q6_K ? (float)w.mult : 0.0f;
            const float mu2 = T == T_Q6_K ? (float)w.mult2 : 0.0f, mm = (float)w.mmin;
#pragma unroll
            for (int n = 0; n < NG; n++) {
                XBlk x;   // token 4 n + i's block; sums where the type needs them
                const uint32_t* xw = (const uint32_t*)(xs + (4 * n + i) * XTOK_ROW + b * Q8_1_BYTES);
                x.d = h2f(xw[0] & 0xFFFFu);
                int lo = 0, sq = 0;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    x.q[e] = (int)xw[1 + e];
                    if (needs_sumq<T>()) (T == T_Q6_K && e < 4 ? lo : sq) = dot4(x.q[e], 0x01010101, T == T_Q6_K && e < 4 ? lo : sq);
                }
                // Q4_0: -8 sum q; Q6_K: -32 sum q of each half
                const int c0 = T == T_Q4_0 ? -8 * sq : T == T_Q6_K ? -32 * lo : 0, c1 = T == T_Q6_K ? -32 * sq : 0;
                v4i s = {c0, c0, c0, c0}, s2 = {c1, c1, c1, c1};
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    if (T == T_Q6_K && e >= 4) s2 = __builtin_amdgcn_mfma_i32_4x4x4i8(w.v[e], x.q[e], s2, 0, 0, 0);
                    else s = __builtin_amdgcn_mfma_i32_4x4x4i8(w.v[e], x.q[e], s, 0, 0, 0);
                }
                auto row_acc = [&](auto rtag) {
                    constexpr int R = decltype(rtag)::value;
                    // the exact block dot: its factors are integers below 2^24
                    float v = (float)s[R];
                    if constexpr (T == T_Q6_K) v = __builtin_fmaf((float)s2[R], quad_of<R>(mu2), v * quad_of<R>(mu));
                    else if constexpr (T == T_IQ3_S || T == T_Q4_K || T == T_Q5_K) v = v * quad_of<R>(mu);
                    float o = __builtin_fmaf(quad_of<R>(w.dw) * x.d, v, acc[n][R]);
                    if constexpr (T == T_Q4_K || T == T_Q5_K)
                        o = __builtin_fmaf(-(quad_of<R>(w.dm) * x.d), quad_of<R>(mm) * (float)sq, o);
                    acc[n][R] = in ? o : acc[n][R];
                };
                row_acc(std::integral_constant<int, 0>{});
                row_acc(std::integral_constant<int, 1>{});
                row_acc(std::integral_constant<int, 2>{});
                row_acc(std::integral_constant<int, 3>{});
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NG; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            // the halving tree over the slots: xor 8, 4, 2, 1 of j
            float v = acc[n][r];
            v = v + xlane<32>(v);
            v = v + xlane<16>(v);
            v = v + xlane<8>(v);
            v = v + xlane<4>(v);
            if (j == 0 && 4 * n + i < a.ntok && 4 * wave + r < nr) a.y[(4 * n + i) * a.y_tok_stride + r0 + 4 * wave + r] = v;
        }
}

// One token, rows of exactly NCH 64-block chunks (2048 * NCH columns), whole
// 16-row tiles, 16-byte aligned rows: the tile's copies, the activation
// blocks, the dots and the L=16 tree with compile-time sizes and a
// compile-time chunk count (the same fp32 order as tile_gemv; the general
// path's run-time row count and chunk loop cost ~0.35 us of latency per
// launch: Q8_0 4096x2048 4.24 -> 3.90 us, Q4_0 head 30.8 -> 28.6 us).
template <int T, int NCH, bool XF32 = false>
__global__ __launch_bounds__(GEMV_THREADS) void k_mmvq_nc(MmvqArgs a) {
    constexpr int CBLK = MMVQ_BLOCKS, CB = chunk_bytes<T>(CBLK), LS = CB + mmvq_pad<T>();
    static_assert(CB % 16 == 0, "16-byte pieces");
    __shared__ __attribute__((aligned(16))) uint8_t tile[TILE_ROWS * LS + 16];
    __shared__ XLds xs[XF32 ? NCH * CBLK : CBLK];
    __shared__ uint32_t grid[T == T_IQ3_S ? 512 : 1];
    const int tid = threadIdx.x, g = tid >> 4, j = tid & 15;
    const int slot = blockIdx.y;
    const int64_t e = a.ids ? (int64_t)a.ids[slot] : (int64_t)slot;
    constexpr int64_t RB = (int64_t)NCH * CB;
    const uint8_t* W = a.W + e * a.w_slot_stride + (int64_t)blockIdx.x * TILE_ROWS * RB;
    const uint8_t* X = a.x + slot * a.x_slot_stride;
    if constexpr (T == T_IQ3_S)
        for (int i = tid; i < 512; i += GEMV_THREADS) grid[i] = c_iq3s_grid_mmvq[i];
    float acc = 0.0f;
#pragma unroll 1
    for (int c = 0; c < NCH; c++) {
        if (c > 0) __syncthreads();   // every wave is done with the previous chunk
        stage_rows_fixed<CB, LS, 16, TILE_ROWS, GEMV_THREADS, CPOL_STREAM, true>(tile, W + c * CB, TILE_ROWS, nullptr,
                                                                                  RB, TILE_ROWS, tid);
        if constexpr (XF32) {
            if (c == 0) {   // the whole row, under the first chunk's copies
                quant_xlds<GEMV_THREADS>((const float*)X, 0, NCH * CBLK, xs, blockIdx.x == 0 ? a.raw : nullptr);
                if (blockIdx.x == 0) raw_padding(a);
            }
        } else if (tid < CBLK) {
            XBlk xb;
            load_xblk(X + (int64_t)(c * CBLK + tid) * Q8_1_BYTES, xb);
            XLds& o = xs[tid];
#pragma unroll
            for (int k = 0; k < 8; k++) o.q[k] = xb.q[k];
            o.d = xb.d;
            o.sumq = T == T_Q4_0S ? (int)xb.sbits : xb.sumq;
        }
        lds_copy_wait();
        __syncthreads();
#pragma unroll 1
        for (int b = j; b < CBLK; b += SLOTS) {
            XBlk xb;
            xlds_to_blk(xs[XF32 ? c * CBLK + b : b], xb);
            WBlk wb;
            block_decode<T>(tile + g * LS, b, grid, wb);
            acc = wacc<T>(wb, xb, acc);
        }
    }
    const float v = slot_reduce16(acc);
    if (j == 0) a.y[slot * a.y_slot_stride + blockIdx.x * TILE_ROWS + g] = v;
}

template <int T, bool XF32 = false>
static void launch_t(const MmvqArgs& a, int nslots, hipStream_t s) {
    dim3 grid((unsigned)((a.nrows + TILE_ROWS - 1) / TILE_ROWS), (unsigned)nslots);
    if constexpr (chunk_bytes<T>(MMVQ_BLOCKS) % 16 == 0) {
        const int nch = a.ncols / (MMVQ_BLOCKS * QK);
        if (a.ntok == 1 && a.ncols % (MMVQ_BLOCKS * QK) == 0 && (nch == 1 || nch == 2) && a.nrows % TILE_ROWS == 0 &&
            (((uintptr_t)a.W | (uintptr_t)a.w_slot_stride) & 15) == 0) {
            if (nch == 1) hipLaunchKernelGGL((k_mmvq_nc<T, 1, XF32>), grid, dim3(GEMV_THREADS), 0, s, a);
            else hipLaunchKernelGGL((k_mmvq_nc<T, 2, XF32>), grid, dim3(GEMV_THREADS), 0, s, a);
            return;
        }
    }
    dim3 blk(GEMV_THREADS);
    if constexpr (XF32) {
        hipLaunchKernelGGL((k_mmvq<T, 1, true>), grid, blk, 0, s, a);
        return;
    }
    if constexpr (T == T_Q4_0S) {   // one token only
        hipLaunchKernelGGL((k_mmvq<T, 1>), grid, blk, 0, s, a);
    } else {
        // k_mmvq_tok works for four tokens at a time: measured (us, k_mmvq /
        // k_mmvq_tok, 151936x2048) 2 tokens Q4_0 30.8 / 39.5, Q6_K 54 / 57; 3
        // tokens Q5_K 47.3 / 48.5; 4 tokens Q4_0 42.7 / 36.7, Q6_K 66 / 55; 5
        // tokens Q4_0 53 / 57, Q5_K 60 / 77; 8 tokens Q8_0 133 / 84, Q4_0 69 /
        // 58, Q5_K 95 / 86, Q6_K 106 / 83, IQ3_S 80 / 64, MXFP4 74 / 61; 7
        // tokens Q4_K 71.8 / 70.4, Q5_K 77 / 85 (16384x4096 21.7 / 23.5, but 4096x2048,
        // one work-group per CU, 8.7 / 8.3)
        constexpr bool KQ = T == T_Q4_K || T == T_Q5_K;
        switch (a.ntok) {
        case 1: hipLaunchKernelGGL((k_mmvq<T, 1>), grid, blk, 0, s, a); break;
        case 2: hipLaunchKernelGGL((k_mmvq<T, 2>), grid, blk, 0, s, a); break;
        case 3: hipLaunchKernelGGL((k_mmvq<T, 3>), grid, blk, 0, s, a); break;
        case 4: hipLaunchKernelGGL((k_mmvq_tok<T, 1>), grid, blk, 0, s, a); break;
        case 5: hipLaunchKernelGGL((k_mmvq<T, 5>), grid, blk, 0, s, a); break;
        case 6:
            if constexpr (KQ) {
                hipLaunchKernelGGL((k_mmvq<T, 6>), grid, blk, 0, s, a);
                break;
            }
            [[fallthrough]];
        case 7:
            if constexpr (T == T_Q5_K)
                if (a.ntok == 7 && grid.x > 256) {
                    hipLaunchKernelGGL((k_mmvq<T, 7>), grid, blk, 0, s, a);
                    break;
                }
            [[fallthrough]];
        default: hipLaunchKernelGGL((k_mmvq_tok<T, 2>), grid, blk, 0, s, a); break;
        }
    }
}

// f32 activation row: x, raw and raw_blocks of a set (k_mmvq)
static void launch_mmvq_f32(int type, const MmvqArgs& a, hipStream_t s) {
    switch (type) {
    case T_Q8_0: launch_t<T_Q8_0, true>(a, 1, s); break;
    case T_Q4_0: launch_t<T_Q4_0, true>(a, 1, s); break;
    case T_IQ3_S: launch_t<T_IQ3_S, true>(a, 1, s); break;
    case T_Q4_K: launch_t<T_Q4_K, true>(a, 1, s); break;
    case T_Q5_K: launch_t<T_Q5_K, true>(a, 1, s); break;
    case T_Q6_K: launch_t<T_Q6_K, true>(a, 1, s); break;
    case T_MXFP4: launch_t<T_MXFP4, true>(a, 1, s); break;
    }
}

bool launch_mmvq(int type, const MmvqArgs& a, int nslots, hipStream_t s) {
    switch (type) {
    case T_Q8_0: launch_t<T_Q8_0>(a, nslots, s); break;
    case T_Q4_0: launch_t<T_Q4_0>(a, nslots, s); break;
    case T_Q4_0S: launch_t<T_Q4_0S>(a, nslots, s); break;
    case T_IQ3_S: launch_t<T_IQ3_S>(a, nslots, s); break;
    case T_Q4_K: launch_t<T_Q4_K>(a, nslots, s); break;
    case T_Q5_K: launch_t<T_Q5_K>(a, nslots, s); break;
    case T_Q6_K: launch_t<T_Q6_K>(a, nslots, s); break;
    case T_MXFP4: launch_t<T_MXFP4>(a, nslots, s); break;
    default: return false;
    }
    return true;
}

// Validates a GEMV request; returns false (error recorded) when rejected.
static bool check_gemv(const char* who, int type, const void* W, const void* x, const float* y,
                       int ncols, int nrows, int nrows_y_padded, int ntok) {
    if (!W || !x || !y) { set_error(CHIMERE_ERR_ARG, "%s: null pointer", who); return false; }
    if (type_block_bytes(type) == 0) {
        set_error(CHIMERE_ERR_ARG, "%s: unsupported type %d", who, type); return false;
    }
    const int elems = type_block_elems(type);
    if (ncols <= 0 || nrows <= 0 || ncols % elems) {
        set_error(CHIMERE_ERR_ARG, "%s: ncols=%d must be a positive multiple of %d (nrows=%d)",
                  who, ncols, elems, nrows);
        return false;
    }
    if (nrows_y_padded < ncols / 32) {
        set_error(CHIMERE_ERR_ARG, "%s: nrows_y_padded=%d < ncols/32=%d", who, nrows_y_padded, ncols / 32);
        return false;
    }
    if (ntok < 1 || ntok > 8) { set_error(CHIMERE_ERR_ARG, "%s: ntok=%d not in 1..8", who, ntok); return false; }
    // MXFP4's 17-byte blocks have no alignment; every other block starts with an f16
    if (((uintptr_t)x & 3) != 0 || (type != T_MXFP4 && ((uintptr_t)W & 1) != 0)) {
        set_error(CHIMERE_ERR_ARG, "%s: Q8_1 input must be 4-byte and weights 2-byte aligned", who);
        return false;
    }
    return true;
}

static void gemv_entry(const char* who, int type, const void* W, const void* x, float* y, int ncols,
                       int nrows, int nrows_y_padded, int ntok, hipStream_t s) {
    // the s-form GEMV reads plain Q4_0 blocks
    if (!check_gemv(who, type == T_Q4_0S ? T_Q4_0 : type, W, x, y, ncols, nrows, nrows_y_padded, ntok)) return;
    MmvqArgs a{(const uint8_t*)W, (const uint8_t*)x, y, ncols, nrows, ntok,
               (int64_t)nrows_y_padded * Q8_1_BYTES, nrows, nullptr, 0, 0, 0, nullptr, 0};
    launch_mmvq(type, a, 1, s);
    check_launch(who);
}

// One launch for an f32 activation row (every work-group quantizes it for
// itself while its first weights are in flight) instead of a quantizer launch
// and the GEMV: the launch costs 1.1-1.4 us per call, the quantizing about
// 0.25 us of vector-ALU time per work-group and 2048 columns.  HIP graph, two
// launches / one: Q8_0 4096x2048 (256 work-groups) 5.4 / 4.5 us, Q5_K 5.4 /
// 4.3; 16384x2048 (1024) Q8_0 10.2 / 9.0, Q4_0 7.9 / 7.1; 65536x2048 (4096)
// Q4_0 16.1 / 17.7; 8192x4096 (512, two chunks) Q5_K 9.5 / 8.8; 16384x4096
// (1024, two chunks) Q5_K 12.2 / 13.1.  Every chunk's quantizing comes before its
// barrier, so rows of many chunks lose again: 2048x6144 (three chunks) Q8_0 10.1 /
// 9.9, Q4_K 8.9 / 8.8, Q6_K 10.1 / 11.3; 2048x8192 (four) Q8_0 12.2 / 12.6, Q5_K 11.1
// / 11.6, Q6_K 12.0 / 14.7.  Not where rows are copied as spans (IQ3_S, Q6_K rows
// off the 16-byte grid): 2048x7168 IQ3_S 15.5 / 15.0, Q6_K 14.6 / 13.9.
// Only where the row, the output and the scratch lie apart: the quantizer launch
// has read all of x before anything is written, so a call may give an output
// (or, for a short row, a scratch) over its input; in one launch other
// work-groups still read x when the first ones store.
static bool f32_one_launch(int type, const float* x, int ncols, int nrows, const float* y, const void* scratch, int ncols_padded) {
    const int64_t wg = (nrows + TILE_ROWS - 1) / TILE_ROWS, chunks = (ncols + MMVQ_BLOCKS * QK - 1) / (MMVQ_BLOCKS * QK);
    const bool spans = (type == T_IQ3_S || type == T_Q6_K) && (row_bytes(type, ncols) & 15) != 0;
    if (wg * chunks > 1024 || (!spans && chunks > (type == T_Q6_K ? 2 : 3))) return false;
    if (((uintptr_t)x & 15) != 0) return false;   // 16-byte loads of x
    auto apart = [](const void* p, int64_t np, const void* q, int64_t nq) {
        return (uintptr_t)p + (uintptr_t)np <= (uintptr_t)q || (uintptr_t)q + (uintptr_t)nq <= (uintptr_t)p;
    };
    const int64_t xb = (int64_t)ncols * 4, yb = (int64_t)nrows * 4, sb = (int64_t)(ncols_padded / QK) * Q8_1_BYTES;
    return apart(x, xb, y, yb) && apart(x, xb, scratch, sb) && apart(y, yb, scratch, sb);
}

static void gemv_f32_entry(const char* who, int type, const void* W, const float* x, float* y,
                           int ncols, int nrows, int ncols_padded, void* scratch, hipStream_t s) {
    if (!x || !scratch) { set_error(CHIMERE_ERR_ARG, "%s: null pointer", who); return; }
    if (ncols_padded < ncols || ncols_padded % 32) {
        set_error(CHIMERE_ERR_ARG, "%s: ncols_padded=%d invalid for ncols=%d", who, ncols_padded, ncols);
        return;
    }
    if (!check_gemv(who, type, W, scratch, y, ncols, nrows, ncols_padded / 32, 1)) return;
    if (f32_one_launch(type, x, ncols, nrows, y, scratch, ncols_padded)) {
        MmvqArgs a{(const uint8_t*)W, (const uint8_t*)x, y, ncols, nrows, 1, 0, nrows, nullptr, 0, 0, 0,
                   (uint8_t*)scratch, ncols_padded / 32};
        launch_mmvq_f32(type, a, s);
        check_launch(who);
        return;
    }
    launch_quantize_q8_1(x, scratch, ncols, ncols_padded, 1, s);
    gemv_entry(who, type, W, scratch, y, ncols, nrows, ncols_padded / 32, 1, s);
}

static void gemv_batched_entry(const char* who, int type, const void* W, const void* x, float* y,
                               const int* ids, int ncols, int nrows, int nrows_y_padded,
                               int64_t expert_stride, int64_t input_stride, int top_k,
                               hipStream_t s) {
    if (!check_gemv(who, type, W, x, y, ncols, nrows, nrows_y_padded, 1)) return;
    if (!ids || top_k <= 0 || expert_stride < row_bytes(type, ncols) * nrows || input_stride < 0 ||
        (input_stride & 3)) {
        set_error(CHIMERE_ERR_ARG, "%s: bad ids/top_k/strides (top_k=%d expert_stride=%lld input_stride=%lld)",
                  who, top_k, (long long)expert_stride, (long long)input_stride);
        return;
    }
    MmvqArgs a{(const uint8_t*)W, (const uint8_t*)x, y, ncols, nrows, 1,
               0, 0, ids, expert_stride, input_stride, nrows, nullptr, 0};
    launch_mmvq(type, a, top_k, s);
    check_launch(who);
}

// ---- debug: exact int32 per-block dots, one thread per (row, block).
// Q4_K / Q5_K: the scaled quant dot sc * sum(q*q_x) (the block's min term is
// m * sum(q_x), a function of the scale bytes and the activation alone).
template <int T>
__global__ void k_block_dots(const uint8_t* __restrict__ W, const uint8_t* __restrict__ x,
                             int32_t* __restrict__ out, int ncols, int nrows) {
    __shared__ uint32_t grid[T == T_IQ3_S ? 512 : 1];
    if constexpr (T == T_IQ3_S)
        for (int i = threadIdx.x; i < 512; i += blockDim.x) grid[i] = c_iq3s_grid_mmvq[i];
    __syncthreads();
    const int nb = ncols / 32;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)nb * nrows) return;
    const int r = (int)(i / nb), b = (int)(i % nb);
    const uint8_t* row = W + (int64_t)r * row_bytes(T, ncols);
    // the block (or its superblock) copied to a private 4-byte aligned buffer
    constexpr int SUPER = QTraits<T>::ELEMS == 256;
    constexpr int LEN = QTraits<T>::BYTES;
    uint8_t buf[(LEN + 7) / 4 * 4] __attribute__((aligned(4)));
    const int64_t off = SUPER ? (int64_t)(b >> 3) * LEN : (int64_t)b * LEN;
    for (int k = 0; k < LEN; k++) buf[k] = row[off + k];
    for (int k = LEN; k < (int)sizeof(buf); k++) buf[k] = 0;
    XBlk xb;
    load_xblk(x + (int64_t)b * Q8_1_BYTES, xb);
    WBlk w;
    block_decode<T>(buf, SUPER ? (b & 7) : 0, grid, w);
    out[i] = wdot<T>(w, xb);
}

template <int T>
static void launch_block_dots(const void* w, const void* x, int32_t* out, int ncols, int nrows, hipStream_t s) {
    const int64_t n = (int64_t)(ncols / 32) * nrows;
    hipLaunchKernelGGL((k_block_dots<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (const uint8_t*)w,
                       (const uint8_t*)x, out, ncols, nrows);
}

}  // namespace chimere

using namespace chimere;

extern "C" {

void chimere_mmvq_iq3s(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, hipStream_t s) {
    gemv_entry("mmvq_iq3s", T_IQ3_S, w, x, y, ncols, nrows, nyp, 1, s);
}
void chimere_mmvq_q8_0(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, hipStream_t s) {
    gemv_entry("mmvq_q8_0", T_Q8_0, w, x, y, ncols, nrows, nyp, 1, s);
}
void chimere_mmvq_q4_0(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, hipStream_t s) {
    gemv_entry("mmvq_q4_0", T_Q4_0, w, x, y, ncols, nrows, nyp, 1, s);
}
void chimere_mmvq_q4_0_sform(const void* w, const void* x, float* y, int ncols, int nrows, int nyp,
                             hipStream_t s) {
    gemv_entry("mmvq_q4_0_sform", T_Q4_0S, w, x, y, ncols, nrows, nyp, 1, s);
}

void chimere_mmvq_iq3s_f32(const void* w, const float* x, float* y, int ncols, int nrows, int ncp,
                           void* scratch, hipStream_t s) {
    gemv_f32_entry("mmvq_iq3s_f32", T_IQ3_S, w, x, y, ncols, nrows, ncp, scratch, s);
}
void chimere_mmvq_q8_0_f32(const void* w, const float* x, float* y, int ncols, int nrows, int ncp,
                           void* scratch, hipStream_t s) {
    gemv_f32_entry("mmvq_q8_0_f32", T_Q8_0, w, x, y, ncols, nrows, ncp, scratch, s);
}
void chimere_mmvq_q4_0_f32(const void* w, const float* x, float* y, int ncols, int nrows, int ncp,
                           void* scratch, hipStream_t s) {
    gemv_f32_entry("mmvq_q4_0_f32", T_Q4_0, w, x, y, ncols, nrows, ncp, scratch, s);
}

void chimere_mmvq_iq3s_batched(const void* w, const void* x, float* y, const int* ids, int ncols,
                               int nrows, int nyp, int64_t es, int64_t is, int top_k, hipStream_t s) {
    gemv_batched_entry("mmvq_iq3s_batched", T_IQ3_S, w, x, y, ids, ncols, nrows, nyp, es, is, top_k, s);
}
void chimere_mmvq_q8_0_batched(const void* w, const void* x, float* y, const int* ids, int ncols,
                               int nrows, int nyp, int64_t es, int64_t is, int top_k, hipStream_t s) {
    gemv_batched_entry("mmvq_q8_0_batched", T_Q8_0, w, x, y, ids, ncols, nrows, nyp, es, is, top_k, s);
}
void chimere_mmvq_q4_0_batched(const void* w, const void* x, float* y, const int* ids, int ncols,
                               int nrows, int nyp, int64_t es, int64_t is, int top_k, hipStream_t s) {
    gemv_batched_entry("mmvq_q4_0_batched", T_Q4_0, w, x, y, ids, ncols, nrows, nyp, es, is, top_k, s);
}

// ggml K-quant / MXFP4 entry points (ffi/ggml_cuda_gemv.cu:118-175, 292-460)
void chimere_mmvq_q5k(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, hipStream_t s) {
    gemv_entry("mmvq_q5k", T_Q5_K, w, x, y, ncols, nrows, nyp, 1, s);
}
void chimere_mmvq_q4k(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, hipStream_t s) {
    gemv_entry("mmvq_q4k", T_Q4_K, w, x, y, ncols, nrows, nyp, 1, s);
}
void chimere_mmvq_q6k(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, hipStream_t s) {
    gemv_entry("mmvq_q6k", T_Q6_K, w, x, y, ncols, nrows, nyp, 1, s);
}
void chimere_mmvq_mxfp4(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, hipStream_t s) {
    gemv_entry("mmvq_mxfp4", T_MXFP4, w, x, y, ncols, nrows, nyp, 1, s);
}
void chimere_mmvq_q5k_f32(const void* w, const float* x, float* y, int ncols, int nrows, int ncp, void* scratch,
                          hipStream_t s) {
    gemv_f32_entry("mmvq_q5k_f32", T_Q5_K, w, x, y, ncols, nrows, ncp, scratch, s);
}
void chimere_mmvq_q4k_f32(const void* w, const float* x, float* y, int ncols, int nrows, int ncp, void* scratch,
                          hipStream_t s) {
    gemv_f32_entry("mmvq_q4k_f32", T_Q4_K, w, x, y, ncols, nrows, ncp, scratch, s);
}
void chimere_mmvq_q6k_f32(const void* w, const float* x, float* y, int ncols, int nrows, int ncp, void* scratch,
                          hipStream_t s) {
    gemv_f32_entry("mmvq_q6k_f32", T_Q6_K, w, x, y, ncols, nrows, ncp, scratch, s);
}
// argument order as the reference's: scratch before the output
void chimere_mmvq_mxfp4_f32(const void* w, const float* x, void* scratch, float* y, int ncols, int nrows, int ncp,
                            hipStream_t s) {
    gemv_f32_entry("mmvq_mxfp4_f32", T_MXFP4, w, x, y, ncols, nrows, ncp, scratch, s);
}
// expert ids are read on the device (the reference dereferences them on the host)
void chimere_mmvq_mxfp4_batched(const void* w, const void* x, float* y, const int* ids, int ncols, int nrows,
                                int nyp, int64_t es, int64_t is, int top_k, hipStream_t s) {
    gemv_batched_entry("mmvq_mxfp4_batched", T_MXFP4, w, x, y, ids, ncols, nrows, nyp, es, is, top_k, s);
}

void chimere_mmvq_multi(int type, const void* w, const void* x, float* y, int ncols, int nrows,
                        int nyp, int ntok, hipStream_t s) {
    gemv_entry("mmvq_multi", type, w, x, y, ncols, nrows, nyp, ntok, s);
}

void chimere_mmvq_q4_0_multi(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, int ntok,
                             hipStream_t s) {
    gemv_entry("mmvq_q4_0_multi", T_Q4_0, w, x, y, ncols, nrows, nyp, ntok, s);
}
void chimere_mmvq_q8_0_multi(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, int ntok,
                             hipStream_t s) {
    gemv_entry("mmvq_q8_0_multi", T_Q8_0, w, x, y, ncols, nrows, nyp, ntok, s);
}
void chimere_mmvq_iq3s_multi(const void* w, const void* x, float* y, int ncols, int nrows, int nyp, int ntok,
                             hipStream_t s) {
    gemv_entry("mmvq_iq3s_multi", T_IQ3_S, w, x, y, ncols, nrows, nyp, ntok, s);
}

void chimere_dbg_block_dots(int type, const void* w, const void* x, int32_t* out, int ncols,
                            int nrows, hipStream_t s) {
    if (!out || !check_gemv("dbg_block_dots", type, w, x, (const float*)out, ncols, nrows, ncols / 32, 1))
        return;
    switch (type) {
    case T_Q8_0: launch_block_dots<T_Q8_0>(w, x, out, ncols, nrows, s); break;
    case T_Q4_0: launch_block_dots<T_Q4_0>(w, x, out, ncols, nrows, s); break;
    case T_IQ3_S: launch_block_dots<T_IQ3_S>(w, x, out, ncols, nrows, s); break;
    case T_Q4_K: launch_block_dots<T_Q4_K>(w, x, out, ncols, nrows, s); break;
    case T_Q5_K: launch_block_dots<T_Q5_K>(w, x, out, ncols, nrows, s); break;
    case T_Q6_K: launch_block_dots<T_Q6_K>(w, x, out, ncols, nrows, s); break;
    case T_MXFP4: launch_block_dots<T_MXFP4>(w, x, out, ncols, nrows, s); break;
    }
    check_launch("dbg_block_dots");
}

}  // extern "C"
