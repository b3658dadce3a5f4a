// gemm_batched.hip — the W8A16 projection for a batch of tokens on the gfx950
// matrix cores, and the paged serving step's fused QKV projection + RoPE +
// paged KV append.
//
//   y[m, n] = sum_k x[m, k] * e4m3(W[n, k]) * scale[n, k / group]
//
// is the reference's w8a16_gemv_kernel (src/kernel/qkv_gemm.cu:32-110) applied
// to each of M tokens: the reference engine decodes one token per step, a
// serving step one per sequence (the paged path's batch). fp32 accumulation,
// fp16 output; the fused form then rotates Q and K (rope.cu:30-45 arithmetic)
// and writes K and V to each token's slot of the paged pool, exactly as
// af_paged_rope_append does on the projection's output.
//
// Every kernel here sums a token's products in one order (a fresh fragment per
// quantisation group, the groups of each of eight parts of K, the parts), so a
// token's result has the same bits whatever launch it is in, from two tokens on.
//
// Few tokens (w8a16_batched_kernel; HBM-bound: one weight byte per 2*M flops, M
// <= 32 per workgroup). Launches of more tokens or rows take the tiled kernel
// further down (pick_tile):
//  * D = X W^T on v_mfma_f32_16x16x32_f16: A = 16 tokens x 32 k of x (read
//    from L2; rows past m repeat row m-1 and are not stored), B = 32 k x 16
//    weight rows (E4M3 -> fp16 in registers with v_cvt_scalef32_pk_f16_fp8 at
//    scale 1, exact). With group sizes that are multiples of 64, a lane loads 16 contiguous weight
//    bytes per pair of MFMAs and the pair's k order is permuted identically on
//    both operands; otherwise 8 bytes per MFMA.
//  * D's column is the lane's weight row, so a group scale is one value per
//    lane: each group accumulates into a fresh fragment, then acc += scale * it.
//  * A workgroup is 8 waves over 16 weight rows: wave p owns the p-th
//    group-aligned part of K, so each workgroup owns its rows' whole K and no
//    partial leaves it. The parts are summed through LDS in a fixed order
//    (results do not depend on timing). 16-row workgroups spread the weights
//    over every CU (320 workgroups for the 5120-row QKV projection); up to 32
//    tokens (two token tiles) share each weight load.
//  * For the fused kernel the 16 columns are 8 head dims d and their rotation
//    partners d + 64, so a pair sits in lanes l and l ^ 8 of a 16-lane row;
//    RoPE runs on the rounded fp16 projections.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "af_common.h"
#include "af_device.h"

namespace af {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2v_t __attribute__((ext_vector_type(2)));

typedef float float4v_t __attribute__((ext_vector_type(4)));
typedef float float16v_t __attribute__((ext_vector_type(16)));

constexpr int kBgParts = 8;               // K parts = waves per workgroup
constexpr int kBgThreads = 64 * kBgParts;  // 512
constexpr int kBgRows = 16;               // weight rows per workgroup (one MFMA column tile)
constexpr int kBgTile = 16;               // tokens per token tile (one MFMA row tile)

struct BatchedArgs {
    const uint16_t* x;  // [m][x_stride] fp16
    int64_t x_stride;
    int m;
    const uint8_t* w;         // [n][k] E4M3
    const uint16_t* scales;   // [n][k / group_size] fp16
    int n, k, group_size, groups;
    uint16_t* y;  // [m][y_stride] fp16 (fused: qkv_out)
    int64_t y_stride;
    // fused paged QKV only
    int n_q_heads, n_kv_heads, head_dim;
    const float* cos_t;
    const float* sin_t;
    int max_pos;
    const int32_t* d_positions;  // [m]
    const int64_t* d_slots;      // [m]
    int64_t max_rows;            // rows of one layer's K (or V) region
    uint8_t* k_dst;              // layer's K region (fp16 or fp8 elements)
    uint8_t* v_dst;
    const float* k_scales;  // fp8 pools: [n_kv_heads]
    const float* v_scales;
    int32_t* d_status;
    // Tiled kernel: y (and in the fused kernel the tables and the pool) allow
    // 16-byte accesses.
    int32_t vec;
};

// Eight E4M3 codes (two dwords) -> eight fp16 values, exact.
__device__ __forceinline__ half8_t e4m3x8(uint32_t lo, uint32_t hi) {
    const half2v_t a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(lo), 1.0f, false);
    const half2v_t b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(lo), 1.0f, true);
    const half2v_t c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(hi), 1.0f, false);
    const half2v_t d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(hi), 1.0f, true);
    return half8_t{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// Weight bytes of one lane for one chunk: 16 (KC = 64) or 8 (KC = 32).
template <int KC>
struct WChunk {
    uint4 v;
};
template <>
struct WChunk<32> {
    uint2 v;
};

// TT token tiles x KC k per chunk; DEPTH chunks in flight per wave.
template <bool FUSED, bool FP8, int TT, int KC>
__global__ __launch_bounds__(kBgThreads, 4) void w8a16_batched_kernel(const BatchedArgs a) {
    constexpr int DEPTH = TT == 1 ? 6 : (KC == 64 ? 2 : 3);  // <= 128 VGPRs: two workgroups per CU
    constexpr int XV = KC / 32;  // 16-byte x loads per token tile per chunk
    __shared__ float s_red[kBgParts][TT * 4][64];
    // KC = 64: each wave's x chunk goes through LDS (see below), 2 KB per token tile.
    __shared__ uint4 s_x[KC == 64 ? kBgParts : 1][TT][2][64];
    __shared__ int32_t s_pos[FUSED ? kBgTile * TT : 1];
    __shared__ int64_t s_slot[FUSED ? kBgTile * TT : 1];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int part = tid >> 6;
    const int j = lane & 15, sub = lane >> 4;  // MFMA column / row index, k sub-block
    const int blk = int(blockIdx.x), t0 = int(blockIdx.y) * kBgTile * TT;
    // The workgroup's 16 weight rows: plain, [16 blk, +16); fused (head_dim 128),
    // dims d0 .. d0+7 of head blk/8 (d0 = 8 (blk % 8)) and their partners d + 64.
    int row;
    if constexpr (FUSED)
        row = (blk >> 3) * 128 + (blk & 7) * 8 + (j & 7) + (j >> 3) * 64;
    else
        row = blk * kBgRows + j;
    const int nrow = min(row, a.n - 1);  // clamped loads

    const int g_lo = part * a.groups / kBgParts, g_hi = (part + 1) * a.groups / kBgParts;
    const int chunks = (g_hi - g_lo) * a.group_size / KC;
    const int per_group = a.group_size / KC;
    const int kbase = g_lo * a.group_size + sub * (KC / 4);  // this lane's first k in a chunk
    const uint8_t* wrow = a.w + size_t(nrow) * a.k + kbase;
    // Token rows past m load row m-1 instead: an MFMA output row depends only on
    // its own A row, and those rows' outputs are never written. (Loading zeros
    // there instead made the compiler select between the x address and a
    // scratch copy of zero, i.e. flat loads, at twice the kernel's time.)
    //
    // KC = 64: x is loaded row-contiguous, not in the MFMA operand layout (which
    // gives the 16 lanes of a k block 16 different token rows, so each load
    // instruction would touch 16 half-used cache lines). Load v of a token tile
    // covers tokens 8v .. 8v+7, one 128-byte line (64 k) per 8 lanes: lane l
    // fetches piece p = (l % 8) ^ ((r / 2) % 8) of token r = 8v + l / 8. The chunk
    // is written to the wave's LDS stage in lane order and read back in operand
    // order; the XOR makes the read of the 16 lanes of a k block hit 16 distinct
    // 16-byte bank groups.
    const uint16_t* xr[TT][KC / 32];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        if constexpr (KC == 64) {
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const int r = 8 * v + (lane >> 3);
                const int piece = (lane & 7) ^ ((r >> 1) & 7);
                const int tok = min(t0 + kBgTile * tt + r, a.m - 1);
                xr[tt][v] = a.x + size_t(tok) * a.x_stride + g_lo * a.group_size + 8 * piece;
            }
        } else {
            const int tok = min(t0 + kBgTile * tt + j, a.m - 1);
            xr[tt][0] = a.x + size_t(tok) * a.x_stride + kbase;
        }
    }

    WChunk<KC> wq[DEPTH];
    uint4 xq[DEPTH][TT][XV];
    uint16_t sq[DEPTH];  // the group scale of each chunk in flight
    const uint16_t* srow = a.scales + size_t(nrow) * a.groups + g_lo;
    auto issue = [&](int slot, int c) __attribute__((always_inline)) {
        sq[slot] = srow[c / per_group];
        if constexpr (KC == 64)
            wq[slot].v = *reinterpret_cast<const uint4*>(wrow + size_t(c) * KC);
        else
            wq[slot].v = *reinterpret_cast<const uint2*>(wrow + size_t(c) * KC);
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int v = 0; v < XV; ++v)
                xq[slot][tt][v] = *reinterpret_cast<const uint4*>(xr[tt][v] + size_t(c) * KC);
    };
#pragma unroll
    for (int i = 0; i < DEPTH; ++i)
        if (i < chunks) issue(i, i);
    if constexpr (FUSED) {  // the tokens' positions and slots, read during the weight stream
        if (tid < kBgTile * TT) {
            const int t = min(t0 + tid, a.m - 1);
            s_pos[tid] = a.d_positions[t];
            s_slot[tid] = a.d_slots[t];
        }
    }

    float4v_t acc[TT], f[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[tt][r] = f[tt][r] = 0.0f;
    for (int c0 = 0; c0 < chunks; c0 += DEPTH) {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) {
            const int c = c0 + i;
            if (c < chunks) {
                const float sc = h2f(sq[i]);
                half8_t wb[XV];
                if constexpr (KC == 64) {
                    wb[0] = e4m3x8(wq[i].v.x, wq[i].v.y);
                    wb[XV - 1] = e4m3x8(wq[i].v.z, wq[i].v.w);
                } else {
                    wb[0] = e4m3x8(wq[i].v.x, wq[i].v.y);
                }
                half8_t xa[TT][XV];
                if constexpr (KC == 64) {
                    // Through the LDS stage: MFMA v takes piece 2 sub + v of token j.
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                        for (int v = 0; v < 2; ++v) {
                            // (a value store: storing the array element directly became a
                            // copy out of private memory and kept xq in scratch)
                            const uint4 val = xq[i][tt][v];
                            s_x[part][tt][v][lane] = make_uint4(val.x, val.y, val.z, val.w);
                        }
                    // The stage writes and reads index one LDS array at run time, so the
                    // compiler keeps their order; the wait orders them in the LDS queue.
                    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                        for (int v = 0; v < 2; ++v) {
                            const int q = 2 * sub + v;
                            const int pos = 8 * (j & 7) + (q ^ ((j >> 1) & 7));
                            xa[tt][v] = __builtin_bit_cast(half8_t, s_x[part][tt][j >> 3][pos]);
                        }
                } else {
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
                        xa[tt][0] = __builtin_bit_cast(half8_t, xq[i][tt][0]);
                }
                if (c + DEPTH < chunks) issue(i, c + DEPTH);  // refill the slot DEPTH chunks ahead
#pragma unroll
                for (int v = 0; v < XV; ++v)
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
                        f[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[tt][v], wb[v], f[tt], 0, 0, 0);
                if ((c + 1) % per_group == 0) {  // group done: scale into the accumulator
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            acc[tt][r] = fmaf(sc, f[tt][r], acc[tt][r]);
                            f[tt][r] = 0.0f;
                        }
                }
            }
        }
    }

    // Sum the parts in a fixed order (part 0 + 1 + ... + 7) through LDS.
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) s_red[part][tt * 4 + r][lane] = acc[tt][r];
    __syncthreads();
    if (part != 0) return;
#pragma unroll
    for (int q = 0; q < TT * 4; ++q) {
        float v = s_red[0][q][lane];
#pragma unroll
        for (int p = 1; p < kBgParts; ++p) v += s_red[p][q][lane];
        acc[q >> 2][q & 3] = v;
    }

    // Register r of token tile tt, lane l: token t0 + 16 tt + 4 (l/16) + r, weight row `row`.
    if constexpr (!FUSED) {
        if (row >= a.n) return;
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = t0 + kBgTile * tt + 4 * sub + r;
                if (t < a.m) a.y[size_t(t) * a.y_stride + row] = f2h(acc[tt][r]);
            }
    } else {
        const int hd = a.head_dim, half = hd / 2;
        const int head = blk >> 3;
        const bool lo = j < 8;               // this lane holds dim d; lane ^ 8 holds d + 64
        const int d = (blk & 7) * 8 + (j & 7);  // pair index, 0 .. 63
        const int dim = lo ? d : d + half;      // the element this lane writes
        const int kind = head < a.n_q_heads ? 0 : (head < a.n_q_heads + a.n_kv_heads ? 1 : 2);
        const int kh = head - a.n_q_heads - (kind == 2 ? a.n_kv_heads : 0);
        const int kv_dim = a.n_kv_heads * hd;
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint16_t mine = f2h(acc[tt][r]);
                const uint16_t other = uint16_t(__shfl_xor(int(mine), 8));
                const int t = t0 + kBgTile * tt + 4 * sub + r;
                if (t >= a.m) continue;
                uint16_t* yrow = a.y + size_t(t) * a.y_stride + size_t(head) * hd;
                const int pos = s_pos[t - t0];
                const int64_t slot = s_slot[t - t0];
                if (pos < 0 || pos >= a.max_pos || slot < 0 || slot >= a.max_rows) {
                    // nothing is rotated or appended for an out-of-range token
                    yrow[dim] = mine;
                    if (a.d_status && j == 0) *a.d_status = AF_ERR_OUT_OF_RANGE;
                    continue;
                }
                const uint16_t y0 = lo ? mine : other, y1 = lo ? other : mine;
                uint16_t o0 = y0, o1 = y1;
                if (kind < 2)
                    rope_rotate(y0, y1, a.cos_t[size_t(pos) * half + d],
                                a.sin_t[size_t(pos) * half + d], o0, o1);
                const uint16_t out = lo ? o0 : o1;
                yrow[dim] = out;
                if (kind > 0) {
                    const size_t e = size_t(slot) * kv_dim + size_t(kh) * hd + dim;
                    uint8_t* base = kind == 1 ? a.k_dst : a.v_dst;
                    if constexpr (FP8) {
                        const float sc = (kind == 1 ? a.k_scales : a.v_scales)[kh];
                        base[e] = uint8_t(quantize_fp8(out, sc));
                    } else {
                        reinterpret_cast<uint16_t*>(base)[e] = out;
                    }
                }
            }
    }
}

// ---- many tokens: a tiled contraction ------------------------------------------
//
// From a few dozen tokens on the projection is no longer the weight stream with a
// little arithmetic: each workgroup re-reads the activations of its tokens (the
// 16-row kernel above reads all of x per 16 rows and the weights once per 32
// tokens), and the matrix cores have work. The tiled kernel gives a workgroup BM
// tokens x BN weight rows; its KS groups of waves take 8 / KS of the eight parts of
// K each, and a wave owns a (BM / WR) x (BN / WC) piece as 32x32x16 MFMAs.
//  * K advances 64 per step. A step's x rows (128 B each, fp16) and weight rows
//    (64 B each, E4M3) go from global memory straight into LDS (lds_dma16), in a
//    ring of ST stages: the loads of step s + ST - 1 are issued in step s, one
//    barrier per step. The weights stay E4M3 in LDS (half the LDS traffic of
//    fp16) and convert in registers, exactly.
//  * 16-byte chunks are XOR-swizzled (x by row / 2, weights by row / 4) so that
//    an operand read of 16 rows covers every bank once; the swizzle is made by
//    choosing which chunk each DMA lane fetches.
//  * The sums are the 16-row kernel's, bit for bit. There, a 16x16x32 MFMA takes
//    bytes 8v .. 8v+7 of each 16 of a 64-k chunk, v = 0 then 1; the hardware adds a
//    16x16x32 product's two halves of K one after the other, exactly as two 32x32x16
//    MFMAs do (compared on random, subnormal, infinite and NaN operands), so a step
//    runs v over both halves of the chunk before the next v. A group's products
//    start from zero, then acc = fma(scale, products, acc), so zero and non-finite
//    scales and activations act as they do there. Parts are added in order, part 0
//    first.
//  * That takes three accumulators per output where K is not cut over waves (group,
//    part, total), and the register file then holds two waves of 64 x 64 per SIMD:
//    2011 tokens of 8192 x 3072 take 109 us (0.93 PFLOP/s; 16-row kernel 432, one
//    rescaled accumulator with four waves per SIMD 101, but its bits depended on the
//    tile), 3072 x 8192 121 (509, 137); 64 tokens of 3072 x 8192 17.2 (26.2, 17.6).
//    With two waves the MFMAs of one run beside the conversions and the fold of the
//    other only in part; issue priority for the wave in its MFMAs is worth 3-5 %.
//  * Group scales: D's column is the lane's weight row, so a group's scale is one
//    value per lane and column tile. Scales are staged in LDS eight groups at a time:
//    a register load waited for in each group would drain the DMA ring with it.
//  * Parts of K on different waves are summed through LDS, and the tile leaves
//    through LDS as fp16, so rows are stored 16 B per lane. In the fused kernel
//    the BN columns are BN / 2 dims d of a head and their partners d + 64, and
//    each thread rotates and appends 8 such pairs of a token from there.
//  * Workgroups are dealt so that each XCD owns whole column panels (its L2
//    then reads each weight once and x once).
constexpr int kScaleChunk = 8;  // groups staged at a time

template <int BM, int BN, int KS, int ST>
struct TileLayout {
    static constexpr int kXBytes = BM * 128;  // one step of x rows
    static constexpr int kWBytes = BN * 64;   // one step of weight rows
    static constexpr int kPart = kXBytes + kWBytes;
    static constexpr int kStage = KS * kPart;
    static constexpr int kRing = ST * kStage;
    static constexpr int kOutStride = BN * 2 + 16;  // bytes between output rows in LDS
    static constexpr int kParts = kBgParts / KS;  // parts of K per wave
    // Sums left for the others: one of the first waves' parts, then each part's.
    static constexpr int kSlots = KS > 1 ? 1 + (KS - 1) * kParts : 0;
    static constexpr int kRed = kSlots * BM * BN * 4;
    static constexpr int kTail = kRed > BM * kOutStride ? kRed : BM * kOutStride;
    static constexpr int kScales = kRing;  // [2][KS][kScaleChunk][BN] fp16 after the ring
    static constexpr int kScaleBytes = ST > 2 ? 2 * KS * kScaleChunk * BN * 2 : 0;
    static constexpr int kLds =
        kRing + kScaleBytes > kTail ? kRing + kScaleBytes : kTail;
};

// The weight row of column c of panel pn: the fused kernel's panels hold dims
// sub * BN / 2 .. of one head (columns below BN / 2) and their rotation partners.
template <bool FUSED, int BN>
__device__ __forceinline__ int panel_row(int pn, int c) {
    if constexpr (!FUSED) return pn * BN + c;
    constexpr int H = BN / 2, SUBS = 64 / H;
    return (pn / SUBS) * 128 + (pn % SUBS) * H + (c % H) + (c / H) * 64;
}

// Stores the tile's fp16 rows from LDS.
template <int BM, int BN, int THREADS, int STRIDE>
__device__ __forceinline__ void store_tile(const BatchedArgs& a, const char* s_out, int t0, int n0,
                                           int tid) {
    constexpr int kChunks = BN / 8;
    for (int c = tid; c < BM * kChunks; c += THREADS) {
        const int r = c / kChunks, q = c % kChunks;
        const int t = t0 + r, col = n0 + 8 * q;
        if (t >= a.m || col >= a.n) continue;
        const uint4 v = *reinterpret_cast<const uint4*>(s_out + r * STRIDE + 16 * q);
        uint16_t* dst = a.y + size_t(t) * a.y_stride + col;
        if (a.vec && col + 8 <= a.n) {
            *reinterpret_cast<uint4*>(dst) = v;
        } else {
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (col + e < a.n) dst[e] = uint16_t(w[e >> 1] >> (16 * (e & 1)));
        }
    }
}

// Rotates the tile's Q and K pairs from LDS, stores them, appends K and V.
template <bool FP8, int BM, int BN, int THREADS, int STRIDE>
__device__ __forceinline__ void store_tile_rope(const BatchedArgs& a, const char* s_out, int t0,
                                                int pn, int tid) {
    constexpr int H = BN / 2, SUBS = 64 / H, kChunks = H / 8;
    const int head = pn / SUBS;
    const int kind = head < a.n_q_heads ? 0 : (head < a.n_q_heads + a.n_kv_heads ? 1 : 2);
    const int kh = head - a.n_q_heads - (kind == 2 ? a.n_kv_heads : 0);
    const int kv_dim = a.n_kv_heads * 128;
    for (int c = tid; c < BM * kChunks; c += THREADS) {
        const int r = c / kChunks, q = c % kChunks;
        const int d = (pn % SUBS) * H + 8 * q;  // pairs (d .. d + 7, d + 64 ..)
        const int t = t0 + r;
        if (t >= a.m) continue;
        const char* row = s_out + r * STRIDE + 16 * q;
        const uint4 vx = *reinterpret_cast<const uint4*>(row);
        const uint4 vy = *reinterpret_cast<const uint4*>(row + 2 * H);
        const uint32_t xw[4] = {vx.x, vx.y, vx.z, vx.w}, yw[4] = {vy.x, vy.y, vy.z, vy.w};
        uint32_t xo[4] = {vx.x, vx.y, vx.z, vx.w}, yo[4] = {vy.x, vy.y, vy.z, vy.w};
        const int pos = a.d_positions[t];
        const int64_t slot = a.d_slots[t];
        // nothing is rotated or appended for an out-of-range token
        const bool ok = pos >= 0 && pos < a.max_pos && slot >= 0 && slot < a.max_rows;
        if (!ok && a.d_status) *a.d_status = AF_ERR_OUT_OF_RANGE;
        if (ok && kind < 2) {
            const float* cr = a.cos_t + size_t(pos) * 64 + d;
            const float* sr = a.sin_t + size_t(pos) * 64 + d;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                uint16_t x0, y0, x1, y1;
                rope_rotate(uint16_t(xw[w]), uint16_t(yw[w]), cr[2 * w], sr[2 * w], x0, y0);
                rope_rotate(uint16_t(xw[w] >> 16), uint16_t(yw[w] >> 16), cr[2 * w + 1],
                            sr[2 * w + 1], x1, y1);
                xo[w] = uint32_t(x0) | (uint32_t(x1) << 16);
                yo[w] = uint32_t(y0) | (uint32_t(y1) << 16);
            }
        }
        auto put = [&](uint16_t* dst, const uint32_t (&v)[4]) {
            if (a.vec) {
                *reinterpret_cast<uint4*>(dst) = make_uint4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) dst[e] = uint16_t(v[e >> 1] >> (16 * (e & 1)));
            }
        };
        uint16_t* yrow = a.y + size_t(t) * a.y_stride + head * 128 + d;
        put(yrow, xo);
        put(yrow + 64, yo);
        if (!ok || kind == 0) continue;
        const size_t e0 = size_t(slot) * kv_dim + size_t(kh) * 128 + d;
        uint8_t* base = kind == 1 ? a.k_dst : a.v_dst;
        if constexpr (FP8) {
            const float sc = (kind == 1 ? a.k_scales : a.v_scales)[kh];
            auto put8 = [&](uint8_t* dst, const uint32_t (&v)[4]) {
                uint32_t code[8];
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    code[e] = quantize_fp8(uint16_t(v[e >> 1] >> (16 * (e & 1))), sc);
                if (a.vec) {
                    *reinterpret_cast<uint2*>(dst) =
                        make_uint2(code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24),
                                   code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24));
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) dst[e] = uint8_t(code[e]);
                }
            };
            put8(base + e0, xo);
            put8(base + e0 + 64, yo);
        } else {
            put(reinterpret_cast<uint16_t*>(base) + e0, xo);
            put(reinterpret_cast<uint16_t*>(base) + e0 + 64, yo);
        }
    }
}

// WGS: workgroups per CU the registers are budgeted for.
template <bool FUSED, bool FP8, int BM, int BN, int WR, int WC, int KS, int ST, int WGS>
__global__ __launch_bounds__(64 * WR * WC * KS, (WGS * WR * WC * KS + 3) / 4) void
w8a16_tiled_kernel(const BatchedArgs a) {
    using L = TileLayout<BM, BN, KS, ST>;
    constexpr int NW = WR * WC, THREADS = 64 * NW * KS;
    constexpr int MT = BM / WR / 32, NT = BN / WC / 32;  // 32x32 tiles of a wave
    constexpr int XI = BM / 8 / NW, WI = BN / 16 / NW;   // DMA instructions of a wave per step
    constexpr int D = ST - 1;           // steps in flight ahead
    // With one step in flight every step waits for all of its wave's loads, so a
    // register load of the next group's scales costs no wait of its own.
    constexpr bool kRegScales = ST == 2;
    static_assert(ST >= 2, "a stage is read while the next one loads");
    static_assert(KS == 1 || kBgParts <= 2 * KS, "a wave keeps at most two parts' sums apart");
    static_assert(MT >= 1 && NT >= 1 && XI >= 1 && WI >= 1, "tile too small for its waves");
    static_assert(XI * 8 * NW == BM && WI * 16 * NW == BN && BN <= 64 * NW, "uneven DMA");
    __shared__ __align__(16) char s_lds[L::kLds];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = KS > 1 ? wid / NW : 0, wave = KS > 1 ? wid % NW : wid;
    const int col = lane & 31, hi = lane >> 5;
    // Tile of this workgroup: workgroup ids go round-robin over the 8 XCDs, so
    // the ids of one XCD take one contiguous range of tiles, token tiles fastest.
    const int mb = (a.m + BM - 1) / BM;
    const int tiles = mb * ((a.n + BN - 1) / BN);
    const int xcd = int(blockIdx.x) & 7, per = tiles >> 3, rest = tiles & 7;
    const int tile = xcd * per + min(xcd, rest) + (int(blockIdx.x) >> 3);
    const int t0 = (tile % mb) * BM, pn = tile / mb;

    // This wave's parts of K, in groups and 64-k steps.
    constexpr int kParts = L::kParts;
    auto part_begin = [&](int p) { return p * a.groups / kBgParts; };
    const int g_lo = part_begin(ks * kParts), g_hi = part_begin((ks + 1) * kParts);
    const int per_group = a.group_size / 64;
    const int steps = (g_hi - g_lo) * per_group;
    const int all_steps = (a.groups + KS - 1) / KS * per_group;  // the longest wave's

    // DMA sources: one scalar base per operand, 32-bit lane offsets. Rows past m
    // or n load the last row: their products are not stored.
    const char* xb = reinterpret_cast<const char*>(a.x + size_t(t0) * a.x_stride) +
                     size_t(g_lo) * a.group_size * 2;
    const int n_first = panel_row<FUSED, BN>(pn, 0);
    const char* wb = reinterpret_cast<const char*>(a.w + size_t(n_first) * a.k) +
                     size_t(g_lo) * a.group_size;
    uint32_t xoff[XI], woff[WI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int r = 8 * (wave * XI + i) + (lane >> 3);
        const int chunk = (lane & 7) ^ ((r >> 1) & 7);
        xoff[i] = uint32_t(min(r, a.m - 1 - t0)) * uint32_t(a.x_stride) * 2u + 16u * chunk;
    }
#pragma unroll
    for (int i = 0; i < WI; ++i) {
        const int r = 16 * (wave * WI + i) + (lane >> 2);
        const int chunk = (lane & 3) ^ ((r >> 2) & 3);
        woff[i] = uint32_t(min(panel_row<FUSED, BN>(pn, r), a.n - 1) - n_first) * uint32_t(a.k) +
                  16u * chunk;
    }
    const uint32_t lds0 = lds_address(s_lds) + ks * L::kPart;
    auto issue = [&](int step, int buf) {
        const uint32_t dst = lds0 + buf * L::kStage;
        const char* xs = xb + size_t(step) * 128;
        const char* ws = wb + size_t(step) * 64;
#pragma unroll
        for (int i = 0; i < XI; ++i) lds_dma16(xs, xoff[i], dst + 1024 * (wave * XI + i));
#pragma unroll
        for (int i = 0; i < WI; ++i)
            lds_dma16(ws, woff[i], dst + L::kXBytes + 1024 * (wave * WI + i));
    };

    // Scales of chunk c (groups g_lo + 8 c ..) of this thread's weight row.
    const int lt = tid - ks * 64 * NW;  // thread within the part
    const bool has_row = lt < BN;
    const uint16_t* srow =
        a.scales + size_t(min(panel_row<FUSED, BN>(pn, min(lt, BN - 1)), a.n - 1)) * a.groups;
    uint16_t* s_scale = reinterpret_cast<uint16_t*>(s_lds + L::kScales);
    uint16_t next_sc[kScaleChunk];
    auto load_scales = [&](int c) {
        if (has_row)
#pragma unroll
            for (int i = 0; i < kScaleChunk; ++i)
                next_sc[i] = srow[min(g_lo + c * kScaleChunk + i, a.groups - 1)];
    };
    auto stage_scales = [&](int c) {
        if (has_row)
#pragma unroll
            for (int i = 0; i < kScaleChunk; ++i)
                s_scale[(((c & 1) * KS + ks) * kScaleChunk + i) * BN + lt] = next_sc[i];
    };
#pragma unroll
    for (int i = 0; i < D; ++i)
        if (i < steps) issue(i, i);
    if constexpr (!kRegScales) {
        load_scales(0);
        stage_scales(0);
        load_scales(1);
    }

    // Operand reads: x row wm + 32 mt + col, weight row wn + 32 nt + col.
    const int wm = (wave / WC) * (BM / WR), wn = (wave % WC) * (BN / WC);
    const int xr = wm + col, wr = wn + col;  // (32 mt does not change (row / 2) % 8)
    uint32_t xa[4], wa[2];
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // q = 2 p + j: 16-byte chunk 4 p + 2 hi + j
        const int chunk = 4 * (q >> 1) + 2 * hi + (q & 1);
        xa[q] = ks * L::kPart + uint32_t(xr) * 128u + 16u * uint32_t(chunk ^ ((xr >> 1) & 7));
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
        wa[p] = ks * L::kPart + L::kXBytes + uint32_t(wr) * 64u +
                16u * uint32_t((2 * p + hi) ^ ((wr >> 2) & 3));

    // f: the current group's products; acc: the current part's sum; done: the sum of
    // the wave's parts before it (one part per wave: unused).
    float16v_t f[MT][NT], acc[MT][NT], done[MT][NT];
    float scale[NT];  // the current group's
    float16v_t zero;
#pragma unroll
    for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        scale[nt] = 0.0f;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) f[mt][nt] = acc[mt][nt] = done[mt][nt] = zero;
    }
    uint16_t sraw[NT];  // kRegScales: the next group's scales
    const uint16_t* slane[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
        slane[nt] = a.scales +
                    size_t(min(panel_row<FUSED, BN>(pn, wr + 32 * nt), a.n - 1)) * a.groups;
        if constexpr (kRegScales) sraw[nt] = slane[nt][min(g_lo, a.groups - 1)];
    }
    // Adds the finished group's products to the part's sum.
    auto fold = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[mt][nt][r] = fmaf(scale[nt], f[mt][nt][r], acc[mt][nt][r]);
    };
    auto end_part = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    done[mt][nt][r] += acc[mt][nt][r];
                    acc[mt][nt][r] = 0.0f;
                }
    };
    using No = std::integral_constant<bool, false>;
    using Yes = std::integral_constant<bool, true>;
    int st = 0, buf = 0;
    // Before step st: its loads have arrived (the D - 1 later steps' may be in
    // flight); the barrier covers the other waves' and frees the buffer read a step
    // ago, which step st + D's loads go to.
    auto arrive = [&]() __attribute__((always_inline)) {
        if (st + D - 1 < steps) wait_vmcnt<(D - 1) * (XI + WI)>();
        else wait_vmcnt<0>();
        __syncthreads();
    };
    auto ahead = [&]() __attribute__((always_inline)) {
        if (st + D < steps) issue(st + D, buf == 0 ? D : buf - 1);
    };
    // One 64-k step; FIRST of a group: the products start from zero.
    auto products = [&](auto first_c) __attribute__((always_inline)) {
        if constexpr (KS == 1) __builtin_amdgcn_s_setprio(1);
        const char* s = s_lds + buf * L::kStage;
        uint4 wv[2][NT];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                wv[p][nt] = *reinterpret_cast<const uint4*>(s + wa[p] + nt * 32 * 64);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                half8_t wf[NT];
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    wf[nt] = j == 0 ? e4m3x8(wv[p][nt].x, wv[p][nt].y)
                                    : e4m3x8(wv[p][nt].z, wv[p][nt].w);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const half8_t xf = __builtin_bit_cast(
                        half8_t,
                        *reinterpret_cast<const uint4*>(s + xa[2 * p + j] + mt * 32 * 128));
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        f[mt][nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                            xf, wf[nt], decltype(first_c)::value && j + p == 0 ? zero : f[mt][nt], 0,
                            0, 0);
                }
            }
        if constexpr (KS == 1) __builtin_amdgcn_s_setprio(0);
        ++st;
        buf = buf == D ? 0 : buf + 1;
    };
    int part = ks * kParts;               // the current part
    int part_end = part_begin(part + 1);  // its last group + 1
    for (int group = g_lo; group < g_hi; ++group) {
        arrive();
        const int gl = group - g_lo;
        if constexpr (!kRegScales)
            if (gl % kScaleChunk == kScaleChunk - 1) {  // read a group later
                const int c = gl / kScaleChunk + 1;
                stage_scales(c);
                load_scales(c + 1);
            }
        ahead();
        fold();
        if (kParts > 1 && group == part_end) {
            end_part();
            do part_end = part_begin(++part + 1);
            while (part_end <= group);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if constexpr (kRegScales) {
                scale[nt] = h2f(sraw[nt]);
                sraw[nt] = slane[nt][min(group + 1, a.groups - 1)];
            } else {
                scale[nt] = h2f(s_scale[((((gl / kScaleChunk) & 1) * KS + ks) * kScaleChunk +
                                         gl % kScaleChunk) * BN + wr + 32 * nt]);
            }
        }
        products(Yes{});
        for (int i = 1; i < per_group; ++i) {
            arrive();
            ahead();
            products(No{});
        }
    }
    for (; st < all_steps; ++st) arrive();  // a wave of fewer steps keeps the others' barriers
    fold();
    if constexpr (KS == 1) end_part();

    // Register r of (mt, nt) is token 32 mt + 8 (r / 4) + 4 hi + r % 4 of the
    // wave's piece, column 32 nt + col.
    __syncthreads();
    auto put = [&](int mt, int nt, int r, float v) {
        const int row = wm + 32 * mt + 8 * (r >> 2) + 4 * hi + (r & 3);
        *reinterpret_cast<uint16_t*>(s_lds + row * L::kOutStride + 2 * (wr + 32 * nt)) = f2h(v);
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 16; ++r) put(mt, nt, r, done[mt][nt][r]);
    } else {
        // The waves of the first parts leave their total in LDS, the others each
        // part's sum; each wave adds up a 16 / KS share of the registers.
        float* red = reinterpret_cast<float*>(s_lds);
        auto at = [&](int slot, int mt, int nt, int r) {
            return ((((slot * NW + wave) * MT + mt) * NT + nt) * 16 + r) * 64 + lane;
        };
        constexpr int RS = 16 / KS;
        float v[MT][NT][RS];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    // (slot 0: the first wave's parts; then part kParts, ..)
                    const int slot = ks == 0 ? 0 : 1 + (ks - 1) * kParts;
                    const float d = done[mt][nt][r], s = acc[mt][nt][r];
                    if (kParts == 1 || ks == 0) {
                        red[at(slot, mt, nt, r)] = kParts == 1 ? s : d + s;
                    } else {
                        red[at(slot, mt, nt, r)] = d;
                        red[at(slot + 1, mt, nt, r)] = s;
                    }
                }
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < RS; ++i) {
                    v[mt][nt][i] = red[at(0, mt, nt, ks * RS + i)];
#pragma unroll
                    for (int q = 1; q < L::kSlots; ++q)
                        v[mt][nt][i] += red[at(q, mt, nt, ks * RS + i)];
                }
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int i = 0; i < RS; ++i) put(mt, nt, ks * RS + i, v[mt][nt][i]);
    }
    __syncthreads();
    if constexpr (FUSED)
        store_tile_rope<FP8, BM, BN, THREADS, L::kOutStride>(a, s_lds, t0, pn, tid);
    else
        store_tile<BM, BN, THREADS, L::kOutStride>(a, s_lds, t0, pn * BN, tid);
}

template <bool FUSED, bool FP8, int BM, int BN, int WR, int WC, int KS, int ST, int WGS>
void launch_tiled(const BatchedArgs& a, hipStream_t s) {
    const int tiles = ((a.m + BM - 1) / BM) * ((a.n + BN - 1) / BN);
    hipLaunchKernelGGL((w8a16_tiled_kernel<FUSED, FP8, BM, BN, WR, WC, KS, ST, WGS>), dim3(tiles),
                       dim3(64 * WR * WC * KS), 0, s, a);
}

// The forms, and what a launch of each was measured to cost on MI355X (eleven
// (n, k) shapes from 4100 x 640 to 14336 x 4096, 2 to 4096 tokens; the model below
// fits each within 3-9 % rms where it is near the best): a round of workgroups,
// `wgs` of them per CU while tiles last, takes `round` plus per 64-k step `step`,
// for each workgroup of the busiest CUs `share` and for each workgroup of the average
// CU `spread` (us); a launch `fixed` besides. Small tiles with several parts of K at a
// time fill the device when tokens or rows are few (their weights and x are then read
// by more workgroups), large ones read the least and keep the matrix cores busiest.
struct TileCost {
    int bm, bn, ks, wgs;
    float fixed, round, step, share, spread;
};
enum { kT128x128, kT64x128, kT64x64, kT64x64k4, kT64x32k4, kT32x64k4, kT32x32k8, kRows16, kRows32,
       kTiles };
constexpr TileCost kTileCost[kTiles] = {
    {128, 128, 1, 2, 1.495f, 10.360f, 0.237f, 0.142f, 0.243f},
    {64, 128, 1, 3, 0.0f, 7.508f, 0.275f, 0.0f, 0.219f},
    {64, 64, 1, 3, 2.463f, 3.766f, 0.148f, 0.048f, 0.089f},
    {64, 64, 4, 1, 3.304f, 2.710f, 0.660f, 0.0f, 0.252f},
    {64, 32, 4, 1, 2.402f, 2.503f, 0.467f, 0.0f, 0.113f},
    {32, 64, 4, 1, 3.203f, 1.723f, 0.477f, 0.0f, 0.159f},
    {32, 32, 8, 1, 3.410f, 1.087f, 0.584f, 0.0f, 0.296f},
    // the 16-row kernel, up to 16 tokens and from 17 on
    {16, 16, 8, 2, 2.584f, 0.0f, 0.156f, 0.403f, 0.203f},
    {32, 16, 8, 4, 3.000f, 0.0f, 0.147f, 0.428f, 0.285f}};

// The cheapest form by kTileCost; kRows16 also for what the tiles do not take: group
// sizes that are not whole 64-k steps and strides past the 32-bit lane offsets. Of the
// measured launches it picks one within 1.3 % of the best on average (17 % at most).
// (us, 16-row kernel / best tile: 3072 rows of k 8192, 16 tokens 14.0 / 15.9, 33 tokens
// 26 / 16.5; 4100 rows of k 640, 16 tokens 4.4 / 5.2; 5120 rows of k 3072, 2 tokens
// 9.9 / 8.6.) All forms give the same bits.
int pick_tile(const BatchedArgs& a) {
    if (a.group_size % 64 != 0 || a.x_stride >= (int64_t(1) << 23) || a.k >= (1 << 24) ||
        int64_t(a.m) * a.n >= (int64_t(1) << 40))
        return kRows16;
    const unsigned cus = unsigned(device_compute_units());
    // (called for every launch: constant tile sizes, 32-bit arithmetic)
    const unsigned m = unsigned(a.m), n = unsigned(a.n), groups = unsigned(a.groups);
    const float per_group = float(a.group_size / 64);
    int best = 0;
    float best_cost = 0.0f;
#pragma clang loop unroll(full)
    for (int i = 0; i < kTiles; ++i) {
        constexpr auto up = [](unsigned x, int by) { return (x + by - 1) / unsigned(by); };
        if (i == (a.m > kBgTile ? kRows16 : kRows32)) continue;
        const TileCost& c = kTileCost[i];
        const unsigned tiles = up(m, c.bm) * up(n, c.bn);  // (m n < 2^40 over 32 x 16 at least)
        const unsigned per_cu = (tiles + cus - 1) / cus;   // shares of the launch's busiest CUs
        const unsigned rounds = up(per_cu, c.wgs);
        const float steps = float(up(groups, c.ks)) * per_group;
        const float cost = c.fixed + float(rounds) * (c.round + steps * c.step) +
                           steps * (float(per_cu) * c.share + float(tiles) / float(cus) * c.spread);
        if (i == 0 || cost < best_cost) {
            best = i;
            best_cost = cost;
        }
    }
    return best;
}

template <bool FUSED, bool FP8>
void launch_tile(int tile, const BatchedArgs& a, hipStream_t s) {
    switch (tile) {
        case kT128x128: return launch_tiled<FUSED, FP8, 128, 128, 2, 2, 1, 3, 2>(a, s);
        case kT64x128: return launch_tiled<FUSED, FP8, 64, 128, 1, 4, 1, 2, 3>(a, s);
        case kT64x64: return launch_tiled<FUSED, FP8, 64, 64, 2, 2, 1, 3, 4>(a, s);
        case kT64x64k4: return launch_tiled<FUSED, FP8, 64, 64, 1, 2, 4, 3, 1>(a, s);
        case kT64x32k4: return launch_tiled<FUSED, FP8, 64, 32, 2, 1, 4, 3, 1>(a, s);
        case kT32x64k4: return launch_tiled<FUSED, FP8, 32, 64, 1, 2, 4, 3, 1>(a, s);
        default: return launch_tiled<FUSED, FP8, 32, 32, 1, 1, 8, 3, 1>(a, s);
    }
}

template <bool FUSED, bool FP8>
void launch_batched(const BatchedArgs& a, int row_blocks, hipStream_t s) {
    const int tile = pick_tile(a);
    if (tile < kRows16) return launch_tile<FUSED, FP8>(tile, a, s);
    const bool two = a.m > kBgTile;
    const int per = kBgTile * (two ? 2 : 1);
    const dim3 grid(row_blocks, (a.m + per - 1) / per), block(kBgThreads);
    const bool k64 = a.group_size % 64 == 0;
    if (two) {
        if (k64) hipLaunchKernelGGL((w8a16_batched_kernel<FUSED, FP8, 2, 64>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((w8a16_batched_kernel<FUSED, FP8, 2, 32>), grid, block, 0, s, a);
    } else {
        if (k64) hipLaunchKernelGGL((w8a16_batched_kernel<FUSED, FP8, 1, 64>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((w8a16_batched_kernel<FUSED, FP8, 1, 32>), grid, block, 0, s, a);
    }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int check_batched(const void* x, int64_t x_stride, int m, const uint8_t* w, const void* scales,
                  int n, int k, int group_size) {
    if (!x || !w || !scales || m < 0 || n <= 0 || k <= 0 || group_size <= 0)
        return AF_ERR_INVALID_ARG;
    if (k % 32 || group_size % 32 || k % group_size) return AF_ERR_UNSUPPORTED;
    if (x_stride < k || x_stride % 8) return AF_ERR_INVALID_ARG;
    if (!aligned16(x) || !aligned16(w)) return AF_ERR_INVALID_ARG;
    return AF_OK;
}

void fill_common(BatchedArgs& a, const void* x, int64_t x_stride, int m, const uint8_t* w,
                 const void* scales, int n, int k, int group_size) {
    a.x = static_cast<const uint16_t*>(x);
    a.x_stride = x_stride;
    a.m = m;
    a.w = w;
    a.scales = static_cast<const uint16_t*>(scales);
    a.n = n;
    a.k = k;
    a.group_size = group_size;
    a.groups = k / group_size;
}

}  // namespace
}  // namespace af

using namespace af;

extern "C" int af_w8a16_gemm_batched(const void* x, int64_t x_stride, int m, const uint8_t* weight,
                                     const void* scales, void* y, int64_t y_stride, int n, int k,
                                     int group_size, af_stream_t stream) {
    if (int st = check_batched(x, x_stride, m, weight, scales, n, k, group_size)) return st;
    if (!y || y_stride < n) return AF_ERR_INVALID_ARG;
    if (m == 0) return AF_OK;
    // One token: the single-token GEMV streams the weights faster than one
    // 16-token MFMA tile that is 15/16 padding.
    if (m == 1) return af_w8a16_gemv(x, weight, scales, y, n, k, group_size, stream);
    BatchedArgs a{};
    fill_common(a, x, x_stride, m, weight, scales, n, k, group_size);
    a.y = static_cast<uint16_t*>(y);
    a.y_stride = y_stride;
    a.vec = aligned16(y) && y_stride % 8 == 0;
    launch_batched<false, false>(a, (n + kBgRows - 1) / kBgRows, static_cast<hipStream_t>(stream));
    AF_TRY_LAUNCH();
    return AF_OK;
}

extern "C" int af_paged_qkv_rope_append(const void* x, int64_t x_stride, int m,
                                        const uint8_t* w_qkv, const void* scales, int k,
                                        int group_size, void* qkv_out, const af_kv_pool* pool,
                                        int layer, const int64_t* d_slots,
                                        const int32_t* d_positions, const float* cos_table,
                                        const float* sin_table, int max_pos, int n_q_heads,
                                        int32_t* d_status, af_stream_t stream) {
    if (!pool || !pool->base || !qkv_out || !d_slots || !d_positions || !cos_table ||
        !sin_table || max_pos <= 0 || n_q_heads <= 0)
        return AF_ERR_INVALID_ARG;
    if (layer < 0 || layer >= pool->n_layers) return AF_ERR_INVALID_ARG;
    if (pool->flags & ~AF_KV_POOL_SHARED_BLOCKS) return AF_ERR_INVALID_ARG;
    const bool fp8 = pool->dtype == AF_KV_FP8_E4M3;
    if (!fp8 && pool->dtype != AF_KV_FP16) return AF_ERR_UNSUPPORTED;
    if (fp8 && !pool->scales) return AF_ERR_INVALID_ARG;
    if (pool->n_kv_heads <= 0) return AF_ERR_INVALID_ARG;
    const int hd = pool->head_dim;
    if (hd != 128) return AF_ERR_UNSUPPORTED;  // a workgroup's columns are d and d + 64
    const int n = (n_q_heads + 2 * pool->n_kv_heads) * hd;
    if (int st = check_batched(x, x_stride, m, w_qkv, scales, n, k, group_size)) return st;
    if (m == 0) return AF_OK;
    const size_t esz = fp8 ? 1 : 2;
    const int kv_dim = pool->n_kv_heads * hd;
    const size_t slab = size_t(pool->total_blocks) * pool->block_size * kv_dim * esz;
    uint8_t* base = static_cast<uint8_t*>(pool->base);
    if (m == 1) {  // one token: the GEMV form, as af_w8a16_gemm_batched at m = 1
        QkvSingleArgs q{};
        q.w = w_qkv;
        q.x = static_cast<const uint16_t*>(x);
        q.scales = static_cast<const uint16_t*>(scales);
        q.k = k;
        q.group_size = group_size;
        q.qkv = static_cast<uint16_t*>(qkv_out);
        q.k_dst = base + size_t(2 * layer) * slab;
        q.v_dst = base + size_t(2 * layer + 1) * slab;
        q.cos_t = cos_table;
        q.sin_t = sin_table;
        q.d_pos = d_positions;
        q.max_pos = max_pos;
        q.d_slot = d_slots;
        q.max_rows = int64_t(pool->total_blocks) * pool->block_size;
        if (fp8) {
            q.k_scales = pool->scales + size_t(layer) * 2 * pool->n_kv_heads;
            q.v_scales = q.k_scales + pool->n_kv_heads;
        }
        q.n_q_heads = n_q_heads;
        q.n_kv_heads = pool->n_kv_heads;
        q.head_dim = hd;
        q.d_status = d_status;
        launch_qkv_single(q, fp8 ? kQkvPagedFp8 : kQkvPagedFp16, static_cast<hipStream_t>(stream));
        AF_TRY_LAUNCH();
        return AF_OK;
    }
    BatchedArgs a{};
    fill_common(a, x, x_stride, m, w_qkv, scales, n, k, group_size);
    a.y = static_cast<uint16_t*>(qkv_out);
    a.y_stride = n;
    a.n_q_heads = n_q_heads;
    a.n_kv_heads = pool->n_kv_heads;
    a.head_dim = hd;
    a.cos_t = cos_table;
    a.sin_t = sin_table;
    a.max_pos = max_pos;
    a.d_positions = d_positions;
    a.d_slots = d_slots;
    a.max_rows = int64_t(pool->total_blocks) * pool->block_size;
    a.k_dst = base + size_t(2 * layer) * slab;
    a.v_dst = base + size_t(2 * layer + 1) * slab;
    if (fp8) {
        a.k_scales = pool->scales + size_t(layer) * 2 * pool->n_kv_heads;
        a.v_scales = a.k_scales + pool->n_kv_heads;
    }
    a.d_status = d_status;
    a.vec = aligned16(qkv_out) && aligned16(cos_table) && aligned16(sin_table) &&
            aligned16(pool->base);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (fp8)
        launch_batched<true, true>(a, n / kBgRows, s);  // eight workgroups per head
    else
        launch_batched<true, false>(a, n / kBgRows, s);
    AF_TRY_LAUNCH();
    return AF_OK;
}
