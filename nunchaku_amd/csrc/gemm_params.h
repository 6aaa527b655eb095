// Kernel argument block and tile constants of the W4A4 GEMM, shared by the host entry point
// (gemm.hip) and the per-variant kernel translation units (gemm_variant.hip).
#pragma once

#include "svdq_common.h"

namespace svdq {


// ranks of the low-rank branch: multiples of 16 up to this (the reference: MAX_RANK = 1024, lora.cuh:22)
constexpr int MAX_RANK = 1024;

constexpr int BM = 256, BN = 256;
// NVFP4 kernel: the operands of one k-group (64 wide) as fp16, dequantized once per workgroup: per operand
// [8 tiles of 32 rows][4 steps of 16 k][2 halves of 8 k][32 rows] x 16 bytes = 32 KB (a wave's fetch of one matrix
// instruction's operand is 1 KB contiguous), activations then weights; two such buffers alternate.
constexpr int OP_BYTES = 8 * 4 * 2 * 32 * 16;    // one operand of one k-group
constexpr int OPBUF_BYTES = 2 * OP_BYTES;          // activations + weights
constexpr int OUT_LD = 136;                // bf16 elements per row of the store-staging slab (128 + pad)
constexpr int SLAB_OFF = 0;                        // 4 waves x (32 rows x OUT_LD bf16): epilogue staging, in the operand buffers' place
static_assert(4 * 32 * OUT_LD * 2 <= 2 * OPBUF_BYTES, "the epilogue's slabs reuse the operand buffers");
// Operands of the low-rank up projection in the epilogue, up to LR_STEPS x 16 ranks: per block of 32 columns (or rows) and 16 ranks 1 KB
// in the order of v_mfma_f32_32x32x16_bf16.  Those of the rows of the waves' first slabs stand where the slabs will.
constexpr int LR_STEPS = 8, LR_BLOCK = LR_STEPS * 1024;
constexpr int LR_UP = 4 * 32 * OUT_LD * 2, LR_ACT = LR_UP + 8 * LR_BLOCK;
static_assert(2 * LR_BLOCK <= LR_UP, "");
__host__ __device__ constexpr int lr_act_block(int wm, int slab) { return slab == 0 ? wm * LR_BLOCK : LR_ACT + ((slab - 1) * 2 + wm) * LR_BLOCK; }
constexpr int TAB_OFF = LR_ACT + 6 * LR_BLOCK;             // 4 waves x float [2][128]: column factors and biases
constexpr int FLAG_OFF = TAB_OFF + 4 * 1024;               // one word: a thread's reading of an arrival counter, for all
// 4 waves: RMS-norm weights of the wave's head, float [128], or the next layer's reciprocal smoothing factors for the wave's columns, float
// [4][NEXT_TAB_LD], 32 of each row used (the lanes of the quantizing pass read the four rows at a time)
constexpr int NEXT_TAB_LD = 36, NEXT_TAB_BYTES = 4 * NEXT_TAB_LD * 4, NEXT_TAB_OFF = FLAG_OFF + 16;
constexpr int LDS_BYTES = NEXT_TAB_OFF + 4 * NEXT_TAB_BYTES;
static_assert(TAB_OFF >= 2 * OPBUF_BYTES, "the tables lie behind the operand buffers");
static_assert(LDS_BYTES <= 160 * 1024, "one workgroup per compute unit");


// Separate q / k / v outputs of a fused QKV projection (EpiloguePackQKV, epilogues.cuh:427-550): fp16
// [heads][rows][128] each, head h at h * head_stride elements.  Rows [attn_tokens, rows) are written with
// the mask value of the tensor: 0 for q and v, NaN for k.
struct QkvOut {
    uint16_t *q, *k, *v;      // null: the epilogue is not composed
    long long stride_q, stride_k, stride_v;
    int attn_tokens, rows;
};

// One wave writes a 32-row x 128-column bf16 slab (one head of q, k or v; rows `ld` elements apart in LDS)
// to the tensor its columns belong to.  Values go bf16 -> fp32 -> fp16 as the reference's convert_half2
// does (epilogues.cuh:446-453); 16 bytes per lane and pass, rows contiguous within a head.
__device__ inline void store_qkv_slab(const QkvOut &o, const uint16_t *slab, int ld, int lane, int row0, int col0, int third) {
    const int which = col0 / third, head = (col0 - which * third) >> 7;
    uint16_t *base = which == 0 ? o.q : (which == 1 ? o.k : o.v);
    const long long stride = which == 0 ? o.stride_q : (which == 1 ? o.stride_k : o.stride_v);
    const uint32_t maskw = which == 1 ? 0x7FFF7FFFu : 0u;  // fp16 NaN pairs for k (epilogues.cuh:543), zeros for q and v
    base += (size_t)head * stride;
#pragma unroll
    for (int pass = 0; pass < 8; pass++) {
        const int rr = pass * 4 + (lane >> 4), cc = (lane & 15) * 8, m = row0 + rr;
        const u32x4_t w = *(const u32x4_t *)(slab + rr * ld + cc);
        u32x4_t d;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const _Float16 lo = (_Float16)bits_f32(w[j] << 16), hi = (_Float16)bits_f32(w[j] & 0xFFFF0000u);
            d[j] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
            if (m >= o.attn_tokens) d[j] = maskw;
        }
        if (m < o.rows) __builtin_nontemporal_store(d, (u32x4_t *)(base + (size_t)m * 128 + cc));
    }
}

// Linear attention (EpilogueLiteLA::apply_litela, epilogues.cuh:572-655).  A wave's 128 output columns are two heads
// of [k 32 | v 32].  vk[i][j] = sum over rows of v[row][i] * relu(k[row][j]) on the matrix cores (the rows are the
// contraction index: both operands are read down the columns of the 32-row bf16 slab in LDS, rows `ld` elements
// apart), row 32 = sum of relu(k[row][j]).  In the INT4 kernel a wave keeps the sums of its slabs in registers
// (VkSums), the two waves of a column half meet in LDS, and the workgroup's row block goes to its own slot of the
// workspace ([row block][head] x 1056 floats, the 32 x 32 part in the lanes' order: a wave's store is 1 KB contiguous);
// the NVFP4 kernel parks every 32-row slab.  A small kernel behind the GEMM adds the row blocks of a batch entry in
// ascending order (reduce_vk_kernel in gemm.hip).
// The reference adds with atomics in the order of arrival (epilogues.cuh:649); atomics here, 2.4 M of them at 4096
// rows and 72 heads, doubled the kernel's time.
constexpr int VK_HEAD_FLOATS = 33 * 32;
struct VkSums {
    float16_t d[2];  // per head: vk[i][j], element e of lane l is i = 8 (e / 4) + 4 (l / 32) + e % 4, j = l % 32
    float ks[2];     // per head: this lane's part of the column sum of relu(k) for j = l % 32
};
__device__ inline void litela_clear(VkSums &s) {
#pragma unroll
    for (int hd = 0; hd < 2; hd++) {
#pragma unroll
        for (int e = 0; e < 16; e++) s.d[hd][e] = 0.f;
        s.ks[hd] = 0.f;
    }
}
__device__ inline void litela_add_slab(VkSums &s, const uint16_t *slab, int ld, int lane) {
    const int j = lane & 31, kb = lane >> 5;
#pragma unroll
    for (int hd = 0; hd < 2; hd++) {
#pragma unroll
        for (int st = 0; st < 2; st++) {
            u32x4_t kw, vw;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                uint32_t kk[2], vv[2];
#pragma unroll
                for (int f = 0; f < 2; f++) {
                    const uint16_t *rowp = slab + (16 * st + 8 * kb + e + f) * ld + hd * 64 + j;
                    kk[f] = rowp[0];
                    vv[f] = rowp[32];
                    if (kk[f] & 0x8000u) kk[f] = 0;  // ReLU on the bf16 value
                    s.ks[hd] += bits_f32(kk[f] << 16);
                }
                kw[e / 2] = kk[0] | (kk[1] << 16);
                vw[e / 2] = vv[0] | (vv[1] << 16);
            }
            s.d[hd] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vw), __builtin_bit_cast(bf16x8_t, kw), s.d[hd], 0, 0, 0);
        }
    }
}
// Writes the wave's two heads to dst (2 x 1056 floats, LDS or the workspace).
template <bool STREAM>
__device__ inline void litela_park(const VkSums &s, float *dst, int lane) {
    const int j = lane & 31, kb = lane >> 5;
#pragma unroll
    for (int hd = 0; hd < 2; hd++) {
        const float ks = s.ks[hd] + __shfl_xor(s.ks[hd], 32);
        float *d = dst + hd * VK_HEAD_FLOATS;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float4_t v = float4_t{s.d[hd][4 * g], s.d[hd][4 * g + 1], s.d[hd][4 * g + 2], s.d[hd][4 * g + 3]};
            if (STREAM) __builtin_nontemporal_store(v, (float4_t *)(d + (g * 64 + lane) * 4));
            else *(float4_t *)(d + (g * 64 + lane) * 4) = v;
        }
        if (kb == 0) d[1024 + j] = ks;
    }
}
// s = s + what another wave parked at src (the rows of s come first).
__device__ inline void litela_add_parked(VkSums &s, const float *src, int lane) {
    const int j = lane & 31, kb = lane >> 5;
#pragma unroll
    for (int hd = 0; hd < 2; hd++) {
        const float ks = s.ks[hd] + __shfl_xor(s.ks[hd], 32);
        const float *d = src + hd * VK_HEAD_FLOATS;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const float4_t v = *(const float4_t *)(d + (g * 64 + lane) * 4);
#pragma unroll
            for (int i = 0; i < 4; i++) s.d[hd][4 * g + i] += v[i];
        }
        s.ks[hd] = kb == 0 ? ks + d[1024 + j] : 0.f;
    }
}
// After the last slab of a tile, called by all four waves (2 x 2, wave = 2 wm + wn) when the tile holds k | v columns
// (a condition uniform over the workgroup): the lower waves hand their sums to the upper ones through their own slab
// areas, which they no longer need, and the upper ones store the row block's share.  `kv`: this wave's columns are k | v.
__device__ inline void litela_finish(VkSums &s, bool kv, int wm, int wn, unsigned char *slabs, int slab_bytes, float *share, int lane) {
    if (kv && wm == 1) litela_park<false>(s, (float *)(slabs + (2 + wn) * slab_bytes), lane);
    __syncthreads();
    if (kv && wm == 0) {
        litela_add_parked(s, (const float *)(slabs + (2 + wn) * slab_bytes), lane);
        litela_park<true>(s, share, lane);
    }
}

struct GemmParams {
    const uint8_t *act;
    const uint16_t *ascales;
    const uint8_t *wgt;
    const _Float16 *wscales;
    const float *colnorm;
    const uint16_t *bias;
    const uint16_t *wcscales;
    const float *lora_act;
    const uint16_t *lora_up;
    uint16_t *out;
    // next-layer fusion
    uint8_t *qout;               // native activation tiles [M_pad, N/2]
    void *oscales;               // bf16 [N/64, M_pad] or fp8 [N/16, M_pad]
    const float *next_smooth_rcp;  // fp32 [N]
    const bf16x8_t *next_down;   // native proj_down of the next layer ([N, R_down])
    float *next_lora_out;        // fp32 [M_pad, R_down], written by the kernel that adds the shares behind the GEMM
    // tiles shared by two workgroups: parked partial sums (fp32 [2 * workgroups][256 threads][64] x 4)
    // and one arrival counter per tile (zero between launches)
    float *partials;
    int *counters;
    int M_pad, N, K, M_out, N_out, R_up, R_down;
    float alpha;
    float lora_scales[MAX_RANK / 16];
    int gelu;
    int silu;  // x * sigmoid(x) before the store (next-layer variants only)
    // RMS norm + rotary embedding on the q and k heads of a fused QKV projection (next-layer variants only)
    const uint16_t *norm_q, *norm_k;  // bf16 [128]
    const float *rotary;              // fp32 [rot_rows/32][16][64 lanes][4], see svdq_gemm_args; null: no such epilogue
    int rot_rows, rope_cols;          // rope_cols = 2 N / 3: the columns of q and k
    float norm_eps;
    QkvOut qkv;
    // linear attention (see g6::Params) and the parked shares of the next layer's low-rank projection
    float *vk, *vk_part;
    int vk_rows;
    int whole_band;              // 0, or (whole tiles only) the band height of the tile numbering in row blocks
    int row_blocks, full_blocks; // few-rows kernels: tiles along M; NVFP4, 64 x 128 tiles: the first so many of 64 rows, the rest of 32 (0: any other launch)
    int lr_steps;                // 16-rank steps of the low-rank operands that are copied to LDS ahead of the main loop
    float *next_lora_part;  // [N/128 column chunks][M_pad/32 slabs][R_down/16][2][64 lanes] x float4
};


// ---- INT4 GEMM on the fp6 matrix instruction (gemm6_kernel.h) -------------------------------------
namespace g6 {
constexpr int BM = 128, BN = 256;  // workgroup tile; 4 waves as 2 x 2, wave tile 64 x 128
// One stage of the LDS ring holds one k-group of the workgroup's operands:
//   4 activation fragments | 8 weight fragments | weight scales 256 x {64 s, 0, 0, 0} bf16 |
//   activation scales 128 x bf16 | zeros (what the upper half-wave reads as its activation scale)
// (tiles of 64 rows: 2 activation fragments, and 1 KB for the activation scales)
template <int MT>
struct StageOf {
    static constexpr int A = 0, W = 2 * MT * FRAG_BYTES, WS = W + 8 * FRAG_BYTES, AS = WS + 256 * 8, Z = AS + (MT == 2 ? 256 : 1024), BYTES = Z + 128;
};
constexpr int STAGE_BYTES = StageOf<2>::BYTES;
static_assert(StageOf<1>::BYTES <= STAGE_BYTES, "both tile heights use the same ring");
constexpr int STAGES = 3;
constexpr int COPIES_PER_WAVE = 6;  // asynchronous copies every wave issues per k-group (128-row tiles)
// epilogue (reuses the ring): per wave one 32-row slab of bf16, then the column tables
constexpr int OUT_LD = 136;
constexpr int SLAB_BYTES = 32 * OUT_LD * 2;
constexpr int EP_TAB = 4 * SLAB_BYTES;     // float cf[256], bias[256]
constexpr int EP_NORMW = EP_TAB + 2048;    // 4 waves x float [128]: RMS-norm weights of the wave's head
constexpr int EP_FLAG = EP_NORMW + 2048;   // one word handed from thread 0 to the workgroup
constexpr int EP_RED = EP_FLAG + 16;       // [2 rank tiles][2 row halves][2][64 lanes] x float4: the two column halves' low-rank sums meet here
constexpr int EP_RED_BYTES = 2 * 2 * 2 * 64 * 16;  // two rank tiles at a time
constexpr int EP_DOWN = EP_RED + EP_RED_BYTES;  // the next layer's proj_down for the tile's 256 columns, up to 2 rank tiles
constexpr int EP_END = EP_DOWN + 16384;
// Before the slabs and the low-rank sums: two chunks of 32 ranks of the low-rank up projection's operands, each
// [256 columns][4 pieces of 16 bytes of lora_up], then [128 rows][8 pieces of 16 bytes of lora_act].  Piece q of a row stands at
// place q ^ swizzle(row): a 16-byte read is served 16 lanes at a time in the order lanes 0-3, 12-15, 20-27, then 4-11, 16-19,
// 28-31, and these 16 rows of 64 (128) bytes then fall on 16 different places of 16 bytes.
constexpr int LR_ACT = 256 * 64, LR_BYTES = LR_ACT + 128 * 128;
constexpr int LR_BUF0 = 0, LR_BUF1 = EP_RED;
static_assert(LR_BUF0 + LR_BYTES <= EP_TAB, "the first chunk lies in the slabs' place");
__host__ __device__ constexpr int lr_up_swizzle(int row) { return (row >> 2) & 3; }
__host__ __device__ constexpr int lr_act_swizzle(int row) { return (row >> 1) & 7; }
constexpr int EP_BYTES = LR_BUF1 + LR_BYTES > EP_END ? LR_BUF1 + LR_BYTES : EP_END;
constexpr int LDS_BYTES = STAGES * STAGE_BYTES > EP_BYTES ? STAGES * STAGE_BYTES : EP_BYTES;
static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups share a compute unit's LDS");

// Which tile a workgroup takes: row blocks [0, full_blocks) are 128 rows high, the half_blocks behind them 64 (or, with
// full_blocks = all, tiles split along K).  Workgroups go to the XCDs round robin (block % 8): each XCD takes one contiguous run of
// the numbers of the 128-row tiles (or their parts), then one of the 64-row tiles'.  The tiles are numbered in bands of about
// ten 128-row blocks, down the band first: the 64 workgroups resident on an XCD at one time then cover about 10 row blocks
// x 6 column blocks, whose operands (6 KB per row block and k-group, 14 KB per column block) they share in that
// XCD's L2.  Measured at 36 x 48 tiles, bytes fetched from beyond the L2 per launch: bands of 6 / 9 / 12 /
// 16 / 18 / 36 row blocks 317 / 296 / 308 / 355 / 396 / 604 MB (the time does not change: 169-171 us).
struct TileOf {
    bool whole;     // 128 rows
    int row_block;  // among the blocks of its height
    int column_block, tile, part;
};
template <typename P>
__host__ __device__ __forceinline__ TileOf tile_of(const P &p, int block, int total, int nblocks) {
    const int full = p.full_blocks * nblocks * p.kparts;
    const int xcd = block % 8, j = block / 8;
    const int first = xcd * (full / 8) + (xcd < full % 8 ? xcd : full % 8);  // of this XCD's 128-row tiles
    const int count = full / 8 + (xcd < full % 8 ? 1 : 0);
    const bool whole = j < count;
    // (the 64-row tiles of the XCDs before this one: their workgroups less their 128-row tiles)
    const int v = whole ? first + j : xcd * (total / 8) + (xcd < total % 8 ? xcd : total % 8) - first + (j - count);
    const int tile = whole ? v / p.kparts : v, part = whole ? v - tile * p.kparts : 0;
    const int blocks = whole ? p.full_blocks : p.half_blocks, band_blocks = whole ? p.band : p.half_band;
    const int band = tile / (band_blocks * nblocks), in_band = tile - band * (band_blocks * nblocks);
    const int rows = blocks - band * band_blocks < band_blocks ? blocks - band * band_blocks : band_blocks;
    const int mb = band * band_blocks + in_band % rows, nb = in_band / rows;
    return TileOf{whole, mb, nb, tile, part};
}
// the height of the bands of `blocks` row blocks: at most `most`, all of the same height where the count allows it
inline int band_height(int blocks, int most) {
    const int bands = (blocks + most - 1) / most;
    return bands > 0 ? (blocks + bands - 1) / bands : 1;
}

struct Params {
    const uint8_t *act;        // fragments [M_pad/128][K/64][4]
    const uint16_t *ascales;   // bf16 [K/64][M_pad]
    const uint8_t *wgt;        // fragments [ceil(N/256)][K/64][8]
    const uint8_t *wscales;    // [ceil(N/256)][K/64][256] x {bf16 64 * scale, 0, 0, 0}
    const uint16_t *bias;      // bf16 [N] or null
    const uint16_t *wcscales;  // bf16 [N] or null
    const float *lora_act;     // fp32 [M_pad][R_up]
    const uint16_t *lora_up;   // bf16 [N][R_up]
    uint16_t *out;             // bf16 [M_out][N_out] or null
    // next-layer fusion
    uint8_t *qout;                 // fragments [M_pad/128][N/64][4] of the next layer's activations
    uint16_t *oscales;             // bf16 [N/64][M_pad]
    const float *next_smooth_rcp;  // fp32 [N]
    const bf16x8_t *next_down;     // native proj_down of the next layer
    float *next_lora_out;          // fp32 [M_pad][R_down]
    float *next_lora_part;         // [N/256 column blocks][M_pad/128][128 x R_down] partial projections, in the lanes' order
    // tiles split along K: parked partial sums and one arrival counter per tile (zero between launches)
    float *partials;
    int *counters;
    // Row blocks of 128 rows, then of 64 rows; and of either kind the row blocks per band of the tile numbering
    int full_blocks, half_blocks, band, half_band;
    int kparts;        // (1 where half_blocks > 0)
    int M_pad, N, K, M_out, N_out, R_up, R_down;
    float alpha;
    float lora_scales[MAX_RANK / 16];
    int gelu, silu;
    const uint16_t *norm_q, *norm_k;
    const float *rotary;
    int rot_rows, rope_cols;
    float norm_eps;
    QkvOut qkv;
    // linear attention (EpilogueLiteLA, epilogues.cuh:552-681; next-layer variant only): columns [0, N/3) are q,
    // stored through `out` after a ReLU; the rest is [head][k 32 | v 32]; vk[batch][head][i][j] += sum over the
    // tile's rows of v[i] relu(k[j]) (i < 32) and of relu(k[j]) (i = 32)
    float *vk;           // fp32 [batch][2 N / 3 / 64][33][32]; null: no such epilogue
    float *vk_part;      // workspace: [full_blocks + half_blocks][heads] x 1056 floats, every row block's sums
    int vk_rows;         // rows per batch entry, a multiple of 256
};
}  // namespace g6

namespace direct {
// The number of the tile that a workgroup of a few-rows launch takes, of `total`.  Workgroups go to the XCDs round robin (number % 8), and each XCD gets one contiguous run of tiles, down the rows
// first, so that the row blocks of a weight column meet in one L2 and every XCD streams its own share of the weights; the 32-row tiles behind 64-row ones likewise.  (A
// function that returns column block and rows too makes the compiler load the kernel's arguments behind the division: 0.2 us a launch.)
__host__ __device__ inline int tile_of(int block, int total) {
    const int xcd = block % 8, extra = total % 8;
    return xcd * (total / 8) + (xcd < extra ? xcd : extra) + block / 8;
}
}  // namespace direct

}  // namespace svdq
