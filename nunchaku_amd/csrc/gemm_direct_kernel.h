// Operator 2 for few rows, INT4 and NVFP4: the same product and epilogues as gemm6_kernel.h and gemm_kernel.h, with
// small output tiles whose operands go from memory straight to the registers of the wave that multiplies them.
//
// The kernels with 128 x 256 and 256 x 256 tiles need thousands of rows to occupy the chip: with a few hundred, a
// layer of N = 3072 is 24 or 12 such tiles, each walking K alone on its compute unit.  Here a workgroup of four waves owns
// a tile of 32 MT rows x 32 NT WN columns; its waves split the columns WN ways and take the k-groups g = part, part + KP, ...
// of their part of K in turn, and the parts' sums meet in LDS at the end.  An operand fragment is contiguous in memory in
// the lanes' order (svdq_common.h), so a wave fetches it with one or two wide loads, DEPTH of its k-groups ahead, and
// neither LDS nor barriers appear in the main loop (but for INT4 tiles whose waves split the columns only and share the rows'
// operands through LDS: STAGED, below).
// What bounds it where compute units have one tile or two: the vector memory path of a compute unit.  It hands out 120 GB/s to requests of
// 16 bytes a lane and 80 to those of 8 (operands in the L2, 48 or 192 compute units at work, 4, 8 or 16 waves each: the same), so that a
// k-group of an INT4 tile of 32 x 128 takes 90 ns, its five fragments 75 of them, and neither more waves nor more k-groups on their way change
// that (eight waves 9.9, three k-groups 9.5 to 10.9 against 8.6 us, M = 256, K = N = 3072).  Plain epilogues therefore choose among six tiles, see
// plain_tile in gemm.hip: square ones fetch least per product, small ones use more compute units.  The others have 128 columns, which a
// head of the norm and a chunk of the next layer's projection have.  With several tiles per compute
// unit the matrix core and the conversions bound it (M = 1157, K = 12288, NVFP4: 10 % waits for operands, 49 and 34 % the others).
// M = 256, K = N = 3072: 22.8 -> 8.8 -> 7.6 us (INT4; 4 us of it do not depend on K), 59.9 -> 10.6 -> 9.2 us (NVFP4); M = 64: 8.6 -> 5.1 and 9.7 -> 5.4.
//
// INT4: one fp6 matrix instruction on the codes, one factor instruction and 16 multiply-adds per 32 x 32 tile and
// k-group (gemm6_kernel.h).  NVFP4: both operands are dequantized to fp16 in registers by the wave that uses them
// (gemm_kernel.h dequantizes once per workgroup; here every wave has its own k-groups, so that is the same).  A wave alone on
// its SIMD issues a vector instruction every 8 cycles at most and stands still behind a matrix instruction while the next one
// waits for the matrix core (32 cycles), so the conversions are counted: 64 rows x 128 columns per wave take 6 of them per matrix
// instruction (64 x 64: 8), converted one step ahead and spread evenly between the matrix instructions (left to itself the
// compiler issues these in pairs, with the conversions behind).  K = 12288, N = 3072, 64 x 64 per wave / 64 x 128 / with the
// conversions a step ahead: M = 256 45.5 / 39.6 / 35.0 us, M = 1157 91.7 / 84.3 / 81.2 (76.4 with buffers, below); from two tiles per compute unit on 1.2
// PFLOP/s, where the large kernel's 1.25 is the power limit.
//
// The epilogue is shared out by columns (tiles narrower than 128: by blocks of 32 x 32): wave w of four adds up the parts' sums of the 32 columns 32 w ... of the tile
// in ascending order, projects the low-rank branch onto them and applies bias, norm, rotation and activation; the
// bf16 tile meets in LDS again and all waves store it, project and quantize it for the next layer.
#pragma once

#include "gemm_math.h"
#include "gemm_params.h"
#include "svdq_quant.h"

namespace svdq {
namespace direct {

template <bool FP4, int MT, int NT>
struct Stage;  // one k-group of a wave's operands on their way from memory
template <int MT, int NT>
struct Stage<false, MT, NT> {
    v6i_t w[NT], x[MT];
    uint32_t ws[NT], as[MT];
};
template <int MT, int NT>
struct Stage<true, MT, NT> {
    u32x4_t w[NT], x[MT];
    uint32_t ws[NT], as[MT];
};

constexpr int SLAB_BYTES = 32 * OUT_LD * 2;
// Waves that split the columns only (WN = 4, INT4, 64 rows): a stage of the rows' operands of one k-group in LDS, two fragments and the scales of
// 64 rows, eight times over in a whole KB; behind them zeros, what the upper half-wave reads as its scale.
constexpr int STAGE_ZEROS = 2 * FRAG_BYTES + 1024, STAGE_BYTES = STAGE_ZEROS + 128;
// LDS.  First the waves' sums, [KP][column tiles (tiles narrower than 128 columns: and row blocks)][4 quads][64 lanes] x float4, 32 rows at a time in tiles of 128 columns,
// or the stages of waves that share the rows' operands; the bf16 slabs take their place, narrow tiles have a slab of its own for every wave behind the sums.  Then the sums of
// squares of the RMS norm, [MT][4][32] floats, and for every wave the factors and biases of its 32 columns.  Beside the stages stand what is copied there while the main loop runs:
// bias and wcscales of the tile's columns, and the low-rank operands of up to LR_AHEAD 16-rank steps, per 32 ranks [columns][4 pieces of 16 bytes of lora_up], then [rows][8 pieces
// of lora_act], piece q of a row at place q ^ swizzle(row) (gemm_params.h).
constexpr int NARROW_LD = 40, NARROW_SLAB_BYTES = 32 * NARROW_LD * 2;
template <int MT, int NT, int WN, int KP, int DEPTH>
struct Lds {
    static constexpr int NC = NT * WN;
    static constexpr bool NARROW = NC < 4, STAGED = KP == 1;
    static constexpr int SUMS = STAGED ? (DEPTH + 1) * STAGE_BYTES : KP * (NARROW ? MT * NC : 4) * 4096;
    static constexpr int SLABS = NARROW ? SUMS : 0, SLABS_END = SLABS + (NARROW ? MT * NC * NARROW_SLAB_BYTES : MT * SLAB_BYTES);
    static constexpr int SSQ = SUMS > SLABS_END ? SUMS : SLABS_END, TAB = SSQ + (NARROW ? 0 : MT * 512), LR = TAB + 4 * 256;  // (beside the stages: bias at TAB, wcscales behind it)
    static constexpr int LR_ACT = NC * 32 * 64, LR_CHUNK = LR_ACT + MT * 32 * 128, LR_AHEAD = STAGED ? 6 : 0;
    // (a compute unit has LDS for two workgroups with six steps ahead or for three with four: M = 256, K = 8064, N = 19840, rank 96, quantizing, 2.4 tiles per compute unit, 80 us
    // with four steps, 87 with six; M = 256, K = 3072, N = 9216, rank 128 22.5 and 20.9)
    static constexpr int lr_steps(int R, bool three) {
        const int most = three && LR_AHEAD > 4 ? 4 : LR_AHEAD;
        return R / 16 < most ? R / 16 : most;
    }
    static constexpr int bytes(int steps) { return LR + (steps + 1) / 2 * LR_CHUNK; }
    static_assert(bytes(LR_AHEAD) <= 80 * 1024 && (!STAGED || 3 * bytes(4) <= 160 * 1024));
};

// The asynchronous copies of the low-rank operands.  A wave's request fetches 16 bytes a lane and fills a KB of LDS in the lanes' order: 16 columns of lora_up, 8 rows of lora_act, of
// 32 ranks (`half`: of the last 16; the other half of the places is then filled with anything).  Where the request's lane reads, from the tile's first column or row and the chunk's first
// rank on (up_base, act_base), and where the multiplying lanes find piece q of a row, counted from the chunk's first column or row.  Used by the host's model of the addresses too.
__host__ __device__ __forceinline__ uint32_t up_copied(int request, int lane, int R, bool half) {
    const int col = request * 16 + (lane >> 2), piece = (lane & 3) ^ g6::lr_up_swizzle(col);
    return (uint32_t)col * (uint32_t)(R * 2) + (half ? piece & 1 : piece) * 16;
}
__host__ __device__ __forceinline__ uint32_t act_copied(int request, int lane, int R, bool half) {
    const int row = request * 8 + (lane >> 3), piece = (lane & 7) ^ g6::lr_act_swizzle(row);
    return (uint32_t)row * (uint32_t)(R * 4) + (half ? piece & 3 : piece) * 16;
}
__host__ __device__ __forceinline__ size_t up_base(int n0, int R, int chunk) { return (size_t)n0 * R * 2 + chunk * 64; }
__host__ __device__ __forceinline__ size_t act_base(int row0, int R, int chunk) { return (size_t)row0 * R * 4 + chunk * 128; }
__host__ __device__ __forceinline__ int up_place(int col, int piece) { return col * 64 + ((piece ^ g6::lr_up_swizzle(col)) << 4); }
__host__ __device__ __forceinline__ int act_place(int row, int piece) { return row * 128 + ((piece ^ g6::lr_act_swizzle(row)) << 4); }

// NVFP4 launches of 64 x 128 tiles have tiles of half the height behind them (few_rows_heights in gemm.hip).
constexpr bool two_heights(bool fp4, int MT, int NC) { return fp4 && MT == 2 && NC == 4; }
// Of NVFP4 tiles of 128 columns the ring of k-groups on their way is as deep as the registers of two waves per SIMD allow (64 rows: a second k-group would fit, and costs 3 % where compute
// units have several tiles).
template <int MT>
constexpr int FP4_RING = MT == 1 ? 2 : 1;

// One tile: MT blocks of 32 rows from block f0 on, column block nb.
// RANKS (NVFP4, tiles of 128 columns, ranks above 32; which launches: copies_ranks in gemm.hip): all four waves need the low-rank operands of the same rows, and a lane that fetches 16 bytes of a row for itself costs
// the vector memory path four times as much as whole pieces of rows do.  The operands go to the place of the sums by asynchronous copies, once these have been
// read, up to rank 128 all at once; two steps requested ahead of the sums and the others behind them, a memory latency each / so, us, the GEMM alone: SiLU, K = 1408, N = 15872, M = 213, rank 64
// 17.4 / 16.3, rank 128 20.4 / 17.5; norm and rotary, M = 505, K = 3072, N = 9216, rank 64 33.9 / 32.3, rank 128 38.9 / 34.1, rank 160 43.0 / 36.1; quantizing, M = 1157, N = 12288, rank 64 100.9 / 98.3,
// rank 128 123.4 / 114.2.  Same bits.  (A kernel of its own: beside the other way in one, ranks up to 32 lost up to 2 %.  INT4: no gain.)
template <bool FP4, int MT, int NT, int WN, int KP, int DEPTH, bool NEXT, bool RANKS>
__device__ __forceinline__ void output_tile(const GemmParams &p, const int nb, const int f0) {
    constexpr int NC = NT * WN;  // 32-column tiles of the workgroup; a wave has NT of them
    constexpr int WAVES = WN * KP;
    constexpr bool NARROW = NC < 4;
    constexpr bool STAGED = WN == 4;
    using L = Lds<MT, NT, WN, KP, DEPTH>;
    static_assert(!STAGED || (!FP4 && MT == 2 && NT == 1 && KP == 1));
    static_assert(WAVES == 4 && MT * NC <= (NARROW ? 4 : 8), "the epilogue gives each wave one column tile, of one row block where the tile is narrow");
    static_assert(!NARROW || !NEXT, "the norm, the rotation and the next layer's operands need whole 128-column blocks");
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r32 = lane & 31, h = lane >> 5;
    const int kgroups = p.K / 64;
    const int kpart = wave / WN, cw = wave % WN;
    const int n0 = nb * (32 * NC);  // first column

    // ---- operands ----------------------------------------------------------------------------------
    // (DEPTH + 1 register sets, indexed by compile-time constants.  The lambdas below reach them through their captures: taken
    // by reference as an argument, a set is known to be readable as a whole, the compiler reads vectors of six words
    // eight wide from it, and then cannot keep it in registers)
    Stage<FP4, MT, NT> sets[DEPTH + 1];
    // The k-group requested next; behind the last one it stays where it is (such a request is never used).
    // INT4: wave-uniform addresses of the operands, which advance by constants.  NVFP4: buffers; a request is a lane's offset that never
    // changes, a scalar one that carries the k-group, and a constant, so that no vector instruction is spent on addresses (21 of 684
    // instructions per three k-groups before): M = 1157, K = 12288, N = 3072 87.4 -> 76.4 us, M = 300, K = N = 3072 10.8 -> 10.6, M = 512, K = 2048,
    // N = 6144 with norm and rotary 22.1 -> 20.0; same bits.  (INT4 with buffers: 8.77 -> 8.99 at M = 256, K = N = 3072, though its loop has a
    // fifth fewer instructions then.)
    int g_load = kpart < kgroups ? kpart : kgroups - 1;
    const uint8_t *wp, *sp, *xp[MT];
    const uint16_t *ap;
    if constexpr (!FP4) {
        constexpr int PER256 = 8 / NC;  // tiles of this width in the 256 columns that the operands are laid out by
        const int blk = nb / PER256, tile0 = nb % PER256 * NC + cw * NT;
        wp = p.wgt + ((size_t)blk * kgroups + g_load) * (8 * FRAG_BYTES) + tile0 * FRAG_BYTES;
        sp = (const uint8_t *)p.wscales + ((size_t)blk * kgroups + g_load) * 2048 + tile0 * 256;
        each(std::make_integer_sequence<int, MT>{}, [&](auto I) {
            constexpr int mt = decltype(I)::value;
            xp[mt] = p.act + ((size_t)((f0 + mt) >> 2) * kgroups + g_load) * (4 * FRAG_BYTES) + ((f0 + mt) & 3) * FRAG_BYTES;
        });
        ap = p.ascales + (size_t)g_load * p.M_pad + f0 * 32;
    }
    const uint32_t off16 = (uint32_t)lane * 16u, off8 = 1024u + (uint32_t)lane * 8u, off_ws = (uint32_t)r32 * 8u + (FP4 ? (uint32_t)h * 4u : 0u);
    const uint32_t off_as = FP4 ? (uint32_t)r32 * 4u + (uint32_t)h * 2u : (uint32_t)r32 * 2u, off_fp4 = (uint32_t)r32 * 32u + (uint32_t)h * 16u;
    const uint32_t tile_stride = (uint32_t)kgroups * TILE_BYTES;  // NVFP4: from one 32-column (or 32-row) tile to the next
    auto buffer = [](const void *base, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, (int)bytes, 0x00020000); };
    const uint32_t s_group = (uint32_t)p.N * 8, a_group = (uint32_t)p.M_pad * 4, s_lead = (n0 + cw * (NT * 32)) * 8, a_lead = f0 * 32 * 4;
    const __amdgpu_buffer_rsrc_t wrsrc = buffer(p.wgt + (size_t)(nb * NC + cw * NT) * kgroups * TILE_BYTES, NT * tile_stride);
    const __amdgpu_buffer_rsrc_t xrsrc = buffer(p.act + (size_t)f0 * kgroups * TILE_BYTES, MT * tile_stride);
    const __amdgpu_buffer_rsrc_t srsrc = buffer((const uint8_t *)p.wscales + s_lead, kgroups * s_group - s_lead);
    const __amdgpu_buffer_rsrc_t arsrc = buffer((const uint8_t *)p.ascales + a_lead, kgroups * a_group - a_lead);
    auto load = [&](auto S) {
        auto &st = sets[decltype(S)::value];
        const bool more = g_load + KP < kgroups;
        if constexpr (FP4) {
            const int o = g_load * TILE_BYTES, so = g_load * (int)s_group, ao = g_load * (int)a_group;
            each(std::make_integer_sequence<int, MT>{}, [&](auto I) {
                constexpr int mt = decltype(I)::value;
                st.x[mt] = __builtin_amdgcn_raw_buffer_load_b128(xrsrc, off_fp4, o + mt * (int)tile_stride, 0);
                st.as[mt] = __builtin_amdgcn_raw_buffer_load_b16(arsrc, off_as + mt * 128, ao, 0);
            });
            each(std::make_integer_sequence<int, NT>{}, [&](auto I) {
                constexpr int nt = decltype(I)::value;
                st.w[nt] = __builtin_amdgcn_raw_buffer_load_b128(wrsrc, off_fp4, o + nt * (int)tile_stride, 0);
                st.ws[nt] = __builtin_amdgcn_raw_buffer_load_b32(srsrc, off_ws + nt * 256, so, 0);
            });
        } else {
            each(std::make_integer_sequence<int, MT>{}, [&](auto I) {
                constexpr int mt = decltype(I)::value;
                st.x[mt] = codes6(*(const u32x4_t *)(xp[mt] + off16), *(const u32x2_t *)(xp[mt] + off8));
                st.as[mt] = *(const uint16_t *)((const uint8_t *)ap + mt * 64 + off_as);
            });
            each(std::make_integer_sequence<int, NT>{}, [&](auto I) {
                constexpr int nt = decltype(I)::value;
                st.w[nt] = codes6(*(const u32x4_t *)(wp + nt * FRAG_BYTES + off16), *(const u32x2_t *)(wp + nt * FRAG_BYTES + off8));
                st.ws[nt] = *(const uint32_t *)(sp + nt * 256 + off_ws);
            });
            wp += more ? KP * 8 * FRAG_BYTES : 0u;
            sp += more ? 2048u * KP : 0u;
            ap += more ? (uint32_t)p.M_pad * KP : 0u;
            each(std::make_integer_sequence<int, MT>{}, [&](auto I) { xp[decltype(I)::value] += more ? KP * 4 * FRAG_BYTES : 0u; });
        }
        g_load += more ? KP : 0;
    };

    // ---- the epilogue's own operands -------------------------------------------------------------------
    // Wave w gets the 32 columns 32 w ... of all MT row blocks; of a narrow tile one of the MT NC blocks of 32 x 32, where there is one.  What it needs for them is requested ahead
    // of the main loop as far as there is room for it: factors and biases; in narrow INT4 tiles the low-rank operands of EARLY 16-rank steps, in registers; beside the stages all of it,
    // in LDS and in whole pieces of rows (a lane that fetches 16 bytes of each of 32 rows for itself costs the vector memory path four times as much).  Requested behind the main loop /
    // as it is, us: INT4 M = 256, K = N = 3072, rank 32 7.84 / 7.55, rank 64 8.8 / 7.9, rank 128 10.0 / 9.3, M = 64 5.24 / 5.01; NVFP4 M = 300 9.3 / 8.9; tiles of 128 columns M = 100,
    // K = 2048, N = 8192, quantizing 15.95 / 15.2, NVFP4 M = 300, K = 3072, N = 9216 with norm and rotary 33.5 / 32.1; shared rows M = 256, K = 3072, N = 9216 with norm and rotary
    // 18.8 / 17.5, rank 128 25.1 / 20.8, quantizing, N = 12288 25.3 / 23.5, M = 200, K = 1024, N = 15360, rank 128 16.2 / 11.6.  Same bits.  Slower: low-rank operands ahead in
    // narrow NVFP4 tiles (several of them share a compute unit: M = 916, K = 1920, N = 1152 10.4 us, 10.7 with), more than two steps in registers, all of them through the place of the
    // sums, which takes two barriers more, the rotary table and the smoothing factors ahead too.  It costs 3 to 4 %
    // where INT4 tiles of 64 x 64 are one to two per compute unit at ranks of 80 and more (M = 600, K = 2048, N = 3200, rank 144 11.5 / 12.0; all such tiles 6 % faster), and 0.1 to 0.2 of 4 us at ranks 16 and 32 with K up
    // to 512 in INT4 tiles of 32 x 64, and of 32 x 32 where there are more than two (all of 32 x 32 6 % faster, of 32 x 64 2).  There too it stays: low-rank operands requested behind the loop's first
    // ones take 4 % of what 32 x 32 tiles gain and 3 % of 32 x 64 ones at rank 0, a branch on K costs 1 to 7 %, and other tiles are no faster.
    constexpr int OWN = NARROW ? 1 : MT, LR_AHEAD = L::LR_AHEAD, EARLY = NARROW && !FP4 ? 2 : 0;
    constexpr bool TABLE = !STAGED && (!NARROW || FP4 || MT * NC < 4);  // factors and biases through a table of the wave's
    const bool owner = !NARROW || wave < MT * NC;
    const int nt = NARROW ? wave % NC : wave, c0 = n0 + nt * 32, row0 = f0 * 32 + (NARROW ? wave / NC * 32 : 0);
    const int nsteps = p.R_up / 16, lr_steps = p.lr_steps;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    struct LowRank {
        float4_t la[OWN][2];
        u32x4_t up;
    };
    auto load_low_rank = [&](LowRank &l, int step) {
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const float4_t *ap = (const float4_t *)(p.lora_act + (size_t)(row0 + o * 32 + r32) * p.R_up + 16 * step + 8 * h);
            l.la[o][0] = ap[0];
            l.la[o][1] = ap[1];
        }
        l.up = *(const u32x4_t *)(p.lora_up + (size_t)(c0 + r32) * p.R_up + 16 * step + 8 * h);
    };
    LowRank early[EARLY > 0 ? EARLY : 1];
    if (owner) {
#pragma unroll
        for (int s = 0; s < EARLY; s++)
            if (nsteps > 0) load_low_rank(early[s], s < nsteps ? s : nsteps - 1);
    }
    // INT4 tiles of 64 x 64 have room for the scales and biases of the lane's columns c0 + 8 q + 4 h + i, the others for those of column c0 + r32.
    constexpr bool RAW = !TABLE && !STAGED;
    u32x2_t wcscales4[RAW ? 4 : 1], bias4[RAW ? 4 : 1];
    float colnorm1 = 1.f;
    uint16_t wcscale1 = 0x3F80, bias1 = 0;
    if constexpr (RAW) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            wcscales4[q] = u32x2_t{0x3F803F80u, 0x3F803F80u};
            bias4[q] = u32x2_t{0u, 0u};
        }
        if (p.wcscales) {
#pragma unroll
            for (int q = 0; q < 4; q++) wcscales4[q] = *(const u32x2_t *)(p.wcscales + c0 + 8 * q + 4 * h);
        }
        if (p.bias) {
#pragma unroll
            for (int q = 0; q < 4; q++) bias4[q] = *(const u32x2_t *)(p.bias + c0 + 8 * q + 4 * h);
        }
    } else if constexpr (TABLE) {
        if (owner) {
            if (FP4) colnorm1 = p.colnorm[c0 + r32];
            if (p.wcscales) wcscale1 = p.wcscales[c0 + r32];
            if (p.bias) bias1 = p.bias[c0 + r32];
        }
    }

    // ---- main loop -----------------------------------------------------------------------------------
    float16_t acc[NT * MT];  // tile t = nt MT + mt
#pragma unroll
    for (int t = 0; t < NT * MT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[t][e] = 0.f;
    // INT4: products and factors of two tiles, one being multiplied while the other is accumulated
    constexpr bool LAG = MT * NT > 1;  // (a single tile per k-group is accumulated at once)
    float16_t P[FP4 ? 1 : 2], F[FP4 ? 1 : 2];
#pragma unroll
    for (int b = 0; b < (FP4 ? 1 : 2); b++)
#pragma unroll
        for (int e = 0; e < 16; e++) P[b][e] = F[b][e] = 0.f;

    // NVFP4: converted operands of two steps, and the rows' scales of the k-group that is being converted
    half8_t wop[FP4 ? 2 : 1], xop[FP4 ? 2 : 1][MT];
    half2_t xs[MT];
    auto column_scale = [](uint32_t ws, bool second) {
        const half2_t s = as_half2(ws);
        return second ? half2_t{s[1], s[1]} : half2_t{s[0], s[0]};
    };
    auto row_scale = [&](int mt, bool second) { return second ? half2_t{xs[mt][1], xs[mt][1]} : half2_t{xs[mt][0], xs[mt][0]}; };
    auto read_row_scales = [&](const uint32_t (&as)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) xs[mt] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(as[mt], 1.0f, false);
    };

    auto compute = [&](auto S) {
        auto &st = sets[decltype(S)::value];
        if constexpr (!FP4) {
            // step t issues the two matrix instructions of tile t and accumulates the tile before it (in the first step the
            // last tile of the k-group before)
            auto tile = [&](auto T) {
                constexpr int t = decltype(T)::value, nt = t / MT, mt = t % MT, b = t & 1, prev = (t + NT * MT - 1) % (NT * MT);
                P[b] = mfma_codes6(st.w[nt], st.x[mt]);
                F[b] = mfma_factor(u32x2_t{st.ws[nt], 0u}, u32x2_t{h ? 0u : st.as[mt], 0u});
#pragma unroll
                for (int e = 0; e < 16; e++) acc[prev][e] = __builtin_fmaf(P[LAG ? b ^ 1 : b][e], F[LAG ? b ^ 1 : b][e], acc[prev][e]);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            each(std::make_integer_sequence<int, NT * MT>{}, tile);
        } else {
            // step t = (ks, nt) multiplies the operands that the step before has converted, and between its matrix instructions
            // converts the column operand of the next step and a share of the rows' operands of the next 16 k (in the last
            // steps those of the next k-group, which arrived while this one was multiplied)
            auto &next = sets[(decltype(S)::value + 1) % (DEPTH + 1)];
            each(std::make_integer_sequence<int, 4 * NT>{}, [&](auto T) {
                constexpr int t = decltype(T)::value, ks = t / NT, nt = t % NT, t1 = (t + 1) % (4 * NT), ks1 = (ks + 1) % 4;
                constexpr bool w_wraps = t1 < t, x_wraps = ks1 < ks;
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[nt * MT + mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wop[t & 1], xop[ks & 1][mt], acc[nt * MT + mt], 0, 0, 0);
                wop[(t + 1) & 1] = dequant_word_fp4((w_wraps ? next : st).w[t1 % NT][t1 / NT], column_scale((w_wraps ? next : st).ws[t1 % NT], t1 / NT >= 2));
                constexpr int share = 4 * MT / NT;  // pairs of the rows' operands per step
                each(std::make_integer_sequence<int, share>{}, [&](auto I) {
                    constexpr int pair = nt * share + decltype(I)::value, mt = pair / 4, b = pair % 4;
                    if constexpr (x_wraps && pair == 0) read_row_scales(next.as);
                    const half2_t v = dequant_pair_fp4<b>((x_wraps ? next : st).x[mt][ks1], row_scale(mt, ks1 >= 2));
                    xop[(ks + 1) & 1][mt][2 * b] = v[0];
                    xop[(ks + 1) & 1][mt][2 * b + 1] = v[1];
                });
                constexpr int valu = (8 + 2 * share + MT - 1) / MT;
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, valu, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        }
    };

    if constexpr (STAGED) {
        // Every wave multiplies one column tile by both row blocks: the columns' operands come straight to registers, DEPTH k-groups ahead, the
        // rows', which all four need, to LDS by asynchronous copies, a KB per wave and k-group, into DEPTH + 1 stages.  Six fragments per
        // k-group and tile where waves that split K two ways fetch eight, no sums to exchange, 32 accumulators per lane.  One tile per compute unit
        // takes 0.2 us per k-group with three on their way (0.33 with two: the latency of the requests), two share it better than that, until the
        // vector instructions bound them: 50 per k-group, with the columns through buffers and the scales as lasting pairs (61 before: QKV M = 256, K =
        // 3072, N = 9216 24.7 -> 23.5 us).  Which launches, and what they gain: staged_rows in gemm.hip.
        const uint32_t base = lds_base + wave * 1024;
        const bool rows = wave < 3;
        const uint8_t *src = rows ? p.act + ((size_t)(f0 >> 2) * kgroups) * (4 * FRAG_BYTES) + (f0 & 3) * FRAG_BYTES + wave * 1024 : (const uint8_t *)(p.ascales + f0 * 32);
        const uint32_t stride = rows ? 4 * FRAG_BYTES : (uint32_t)p.M_pad * 2, voff = rows ? lane * 16 : (lane & 7) * 16;
        constexpr int RING = DEPTH + 1;
        v6i_t w[RING];
        u32x2_t ws[RING], as[MT];  // (pairs whose second register stays zero: opaque, so that it is not made again with every scale)
#pragma unroll
        for (int i = 0; i < RING; i++) {
            ws[i] = u32x2_t{0u, 0u};
            asm volatile("" : "+v"(ws[i]));
        }
#pragma unroll
        for (int i = 0; i < MT; i++) {
            as[i] = u32x2_t{0u, 0u};
            asm volatile("" : "+v"(as[i]));
        }
        if (threadIdx.x < RING * 32) *(uint32_t *)(lds + (threadIdx.x >> 5) * STAGE_BYTES + STAGE_ZEROS + (threadIdx.x & 31) * 4) = 0u;
        const uint32_t off_rows = h ? (uint32_t)STAGE_ZEROS : 2u * FRAG_BYTES + (uint32_t)r32 * 2u;
        const __amdgpu_buffer_rsrc_t wbuf = buffer(wp, (uint32_t)(kgroups - 1) * (8 * FRAG_BYTES) + FRAG_BYTES), sbuf = buffer(sp, (uint32_t)(kgroups - 1) * 2048 + 256);
        int g_req = 0;
        // The epilogue's operands: the oldest requests, landed when the first k-group has, with all others' behind the same barrier.  (Code of its own behind the kernel's.)
        if (__builtin_expect(lr_steps > 0 || p.bias || p.wcscales, 0)) {
            const uint8_t *columns = (const uint8_t *)(wave == 0 ? p.bias : wave == 1 ? p.wcscales : nullptr);  // 128 bf16: a word a lane
            if (columns)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" :: "s"(lds_base + L::TAB + wave * 256), "v"(lane * 4), "s"(columns + n0 * 2) : "memory", "m0");
            // (32 ranks at a time; which 16 bytes of its row a lane fetches is permuted as in gemm6_kernel.h)
            for (int c = 0; 2 * c < lr_steps; c++) {
                const bool half = nsteps - 2 * c < 2;
                const uint32_t place = lds_base + L::LR + c * L::LR_CHUNK;
                const uint8_t *up = (const uint8_t *)p.lora_up + up_base(n0, p.R_up, c), *la = (const uint8_t *)p.lora_act + act_base(row0, p.R_up, c);
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const uint32_t up_off = up_copied(wave * 2 + i, lane, p.R_up, half), act_off = act_copied(wave * 2 + i, lane, p.R_up, half);
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(place + (wave * 2 + i) * 1024), "v"(up_off), "s"(up) : "memory", "m0");
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(place + L::LR_ACT + (wave * 2 + i) * 1024), "v"(act_off), "s"(la) : "memory", "m0");
                }
            }
        }
        auto request = [&](auto S) {
            constexpr int st = decltype(S)::value;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(base + st * STAGE_BYTES), "v"(voff), "s"(src) : "memory", "m0");
            w[st] = codes6(__builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wbuf, off16, g_req * (8 * FRAG_BYTES), 0)),
                           __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(wbuf, off8, g_req * (8 * FRAG_BYTES), 0)));
            ws[st][0] = __builtin_amdgcn_raw_buffer_load_b32(sbuf, off_ws, g_req * 2048, 0);
            src += stride;
            g_req++;
        };
        v6i_t X[MT];
        auto read_rows = [&](auto S) {
            const uint8_t *stage = lds + decltype(S)::value * STAGE_BYTES;
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                X[mt] = codes6(*(const u32x4_t *)(stage + mt * FRAG_BYTES + off16), *(const u32x2_t *)(stage + mt * FRAG_BYTES + off8));
                as[mt][0] = *(const uint16_t *)(stage + mt * 64 + off_rows);
            }
        };
        // A wave's copy of a k-group has landed once no more requests are left than were made after it: three for its columns, then a copy and three more
        // for every k-group requested behind it (each of them is used, so that the compiler drops none; what it waits for its own loads with
        // does not count the copies and is stricter).  All waves' copies have landed behind the barrier.
        auto landed = [&](auto BEHIND) { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(3 + 4 * decltype(BEHIND)::value) : "memory"); };
        // A k-group and the LEFT that follow it and are requested by its end (DEPTH: one more is requested here)
        auto body = [&](auto S, auto LEFT) {
            constexpr int st = decltype(S)::value, left = decltype(LEFT)::value;
            // (the stage was that of the k-group before this one, read before the last barrier)
            if constexpr (left == DEPTH) request(std::integral_constant<int, (st + DEPTH) % RING>{});
            __builtin_amdgcn_sched_barrier(0);
            // the first tile's instructions, and between them the additions of the second one of the k-group before
            auto add = [&](int mt) {
#pragma unroll
                for (int e = 0; e < 16; e++) acc[mt][e] = __builtin_fmaf(P[mt][e], F[mt][e], acc[mt][e]);
            };
            P[0] = mfma_codes6(w[st], X[0]);
            F[0] = mfma_factor(ws[st], as[0]);
            add(1);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 9, 0);
            __builtin_amdgcn_sched_barrier(0);
            P[1] = mfma_codes6(w[st], X[1]);
            F[1] = mfma_factor(ws[st], as[1]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (left > 0) {
                landed(std::integral_constant<int, left - 1>{});
                read_rows(std::integral_constant<int, (st + 1) % RING>{});
            }
            add(0);
            if constexpr (left == 0) add(1);
            __builtin_amdgcn_sched_barrier(0);
        };
        // What whole turns of the ring leave over of the k-groups before the last DEPTH comes first: the register sets at the end are then the same
        // ones whatever their number (an end for each carried the accumulators through scratch memory).
        constexpr std::integral_constant<int, DEPTH> ALL;
        auto start = [&](auto ODD) {
            constexpr int odd = decltype(ODD)::value;
            each(std::make_integer_sequence<int, DEPTH>{}, [&](auto I) { request(std::integral_constant<int, (decltype(I)::value + RING - odd) % RING>{}); });
            landed(std::integral_constant<int, DEPTH - 1>{});
            read_rows(std::integral_constant<int, (RING - odd) % RING>{});
            each(std::make_integer_sequence<int, odd>{}, [&](auto I) { body(std::integral_constant<int, (decltype(I)::value + RING - odd) % RING>{}, ALL); });
        };
        // (kgroups > DEPTH, and even: K is a multiple of 128.  So one or three are left over.)
        static_assert(RING == 4);
        const int odd = (kgroups - DEPTH) % RING;
        if (odd == 1) start(std::integral_constant<int, 1>{});
        else start(std::integral_constant<int, 3>{});
        for (int g = odd; g + DEPTH < kgroups; g += RING) each(std::make_integer_sequence<int, RING>{}, [&](auto I) { body(I, ALL); });
        each(std::make_integer_sequence<int, DEPTH>{}, [&](auto I) { body(I, std::integral_constant<int, DEPTH - 1 - decltype(I)::value>{}); });
        // (the sums are wanted here: the compiler would move the last additions behind the epilogue's requests, and their operands to scratch memory)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int e = 0; e < 16; e++) asm volatile("" : "+v"(acc[mt][e]));
        __syncthreads();  // everybody has read the last stage: the slabs take the stages' place
    } else {
        each(std::make_integer_sequence<int, DEPTH>{}, [&](auto D) { load(D); });
        if constexpr (FP4) {
            auto &st = sets[0];
            read_row_scales(st.as);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) xop[0][mt] = dequant_word_fp4(st.x[mt][0], row_scale(mt, false));
            wop[0] = dequant_word_fp4(st.w[0][0], column_scale(st.ws[0], false));
        }
        int g = kpart;
        auto step = [&](auto S) {
            load(std::integral_constant<int, (decltype(S)::value + DEPTH) % (DEPTH + 1)>{});
            __builtin_amdgcn_sched_barrier(0);
            compute(S);
            g += KP;
        };
        // (whole turns of the ring in the loop, what is left behind it: leaving the loop in the middle of a turn makes the
        // compiler carry two copies of the accumulators)
        while (g + DEPTH * KP < kgroups) each(std::make_integer_sequence<int, DEPTH + 1>{}, step);
        if (g < kgroups) step(std::integral_constant<int, 0>{});
        if constexpr (DEPTH > 1) {
            if (g < kgroups) step(std::integral_constant<int, 1>{});
        }
        if constexpr (DEPTH > 2) {
            if (g < kgroups) step(std::integral_constant<int, 2>{});
        }
        if constexpr (!FP4 && LAG) {
#pragma unroll
            for (int e = 0; e < 16; e++) acc[NT * MT - 1][e] = __builtin_fmaf(P[1][e], F[1][e], acc[NT * MT - 1][e]);
        }
    }

    // The low-rank operands that have not been requested yet, two steps at a time (four, three of two row blocks or six in narrow tiles: slower).
    constexpr int LSTEPS = 2;
    const int LFIRST = STAGED ? lr_steps : EARLY;
    LowRank more[LSTEPS];
    auto load_more = [&](int s0) {
#pragma unroll
        for (int s = 0; s < LSTEPS; s++) load_low_rank(more[s], s0 + s < nsteps ? s0 + s : nsteps - 1);  // (a request behind a branch makes the compiler wait for those before it)
    };
    static_assert(!RANKS || (!NARROW && !STAGED && KP == 4));
    constexpr int COPIED = RANKS ? 2 * (L::SUMS / L::LR_CHUNK) : 0;  // steps that the place of the sums holds
    const int copied = nsteps < COPIED ? nsteps : COPIED;
    if (!RANKS && owner && LFIRST < nsteps) load_more(LFIRST);
    // Factor and bias of the lane's columns c0 + 8 q + 4 h + i.
    float *tab = (float *)(lds + L::TAB + wave * 256);
    if (TABLE && h == 0) {
        tab[r32] = colnorm1 * p.alpha * bf16_bits_to_f32(wcscale1);
        tab[32 + r32] = bf16_bits_to_f32(bias1);
    }
    auto four = [](u32x2_t w) {
        return float4_t{bits_f32(w[0] << 16), bits_f32(w[0] & 0xFFFF0000u), bits_f32(w[1] << 16), bits_f32(w[1] & 0xFFFF0000u)};
    };
    auto factors = [&](int q) {
        if constexpr (TABLE) return *(const float4_t *)(tab + 8 * q + 4 * h);
        float4_t f = {1.f, 1.f, 1.f, 1.f}, w;
        if constexpr (STAGED) {
            w = p.wcscales ? four(*(const u32x2_t *)(lds + L::TAB + 256 + (nt * 32 + 8 * q + 4 * h) * 2)) : f;
        } else {
            w = four(wcscales4[q]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) f[i] = f[i] * p.alpha * w[i];
        return f;
    };
    auto biases = [&](int q) {
        if constexpr (TABLE) return *(const float4_t *)(tab + 32 + 8 * q + 4 * h);
        else if constexpr (STAGED) return p.bias ? four(*(const u32x2_t *)(lds + L::TAB + (nt * 32 + 8 * q + 4 * h) * 2)) : float4_t{0.f, 0.f, 0.f, 0.f};
        else return four(bias4[q]);
    };

    // ---- the waves' sums meet, 32 rows at a time, added in ascending order of the waves ---------------------
    float16_t val[OWN];
    float4_t *park = (float4_t *)lds;
    if constexpr (STAGED) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) val[mt] = acc[mt];
    } else if constexpr (NARROW) {
#pragma unroll
        for (int t = 0; t < NT * MT; t++) {
            const int tile = t % MT * NC + cw * NT + t / MT;
#pragma unroll
            for (int q = 0; q < 4; q++)
                park[((kpart * (MT * NC) + tile) * 4 + q) * 64 + lane] = float4_t{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
        }
        __syncthreads();
        if (!owner) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float4_t s = park[(wave * 4 + q) * 64 + lane];
#pragma unroll
            for (int j = 1; j < KP; j++) s += park[((j * (MT * NC) + wave) * 4 + q) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; i++) val[0][4 * q + i] = s[i];
        }
    } else {
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            if (mt > 0) __syncthreads();
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    park[((kpart * 4 + cw * NT + t) * 4 + q) * 64 + lane] =
                        float4_t{acc[t * MT + mt][4 * q], acc[t * MT + mt][4 * q + 1], acc[t * MT + mt][4 * q + 2], acc[t * MT + mt][4 * q + 3]};
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float4_t s = park[(nt * 4 + q) * 64 + lane];
#pragma unroll
                for (int j = 1; j < KP; j++) s += park[((j * 4 + nt) * 4 + q) * 64 + lane];
#pragma unroll
                for (int i = 0; i < 4; i++) val[mt][4 * q + i] = s[i];
            }
        }
        __syncthreads();  // the sums have been read: the low-rank operands (RANKS) and then the slabs take their place
        // (32 ranks at a time; which 16 bytes of its row a lane fetches is permuted as in gemm6_kernel.h)
        for (int c = 0; 2 * c < copied; c++) {
            const bool half = nsteps - 2 * c < 2;
            const uint32_t place = lds_base + c * L::LR_CHUNK;
            const uint8_t *up = (const uint8_t *)p.lora_up + up_base(n0, p.R_up, c), *la = (const uint8_t *)p.lora_act + act_base(row0, p.R_up, c);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t up_off = up_copied(wave * 2 + i, lane, p.R_up, half);
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(place + (wave * 2 + i) * 1024), "v"(up_off), "s"(up) : "memory", "m0");
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const uint32_t act_off = act_copied(wave * MT + i, lane, p.R_up, half);
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(place + L::LR_ACT + (wave * MT + i) * 1024), "v"(act_off), "s"(la) : "memory", "m0");
            }
        }
    }

    float *ssq = (float *)(lds + L::SSQ);  // [MT][4 column tiles][32 rows]
    const bool rope = NEXT && p.rotary && n0 < p.rope_cols;  // the tile is one head of q or k
    if (FP4 || p.wcscales || p.alpha != 1.f) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float4_t cf = factors(q);
#pragma unroll
            for (int o = 0; o < OWN; o++)
#pragma unroll
                for (int i = 0; i < 4; i++) val[o][4 * q + i] *= cf[i];
        }
    }
    // Low-rank up projection (lora.cuh:110-241): out += bf16(lora_act * scale) @ up^T
    auto add_low_rank = [&](int o, int step, float4_t v0, float4_t v1, u32x4_t up) {
        const float ls = p.lora_scales[step];
        u32x4_t w;
        w[0] = pack_bf16x2(v0[0] * ls, v0[1] * ls);
        w[1] = pack_bf16x2(v0[2] * ls, v0[3] * ls);
        w[2] = pack_bf16x2(v1[0] * ls, v1[1] * ls);
        w[3] = pack_bf16x2(v1[2] * ls, v1[3] * ls);
        val[o] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, up), __builtin_bit_cast(bf16x8_t, w), val[o], 0, 0, 0);
    };
    auto add_step = [&](const LowRank &l, int step) {
#pragma unroll
        for (int o = 0; o < OWN; o++) add_low_rank(o, step, l.la[o][0], l.la[o][1], l.up);
    };
#pragma unroll
    for (int s = 0; s < EARLY; s++)
        if (s < nsteps) add_step(early[s], s);
    auto add_copied = [&](const uint8_t *chunk, int s) {
        const uint8_t *buf = chunk + (s / 2) * L::LR_CHUNK;
        const int col = wave * 32 + r32, k = s % 2;
        const u32x4_t up = *(const u32x4_t *)(buf + up_place(col, 2 * k + h));
#pragma unroll
        for (int o = 0; o < OWN; o++) {
            const int row = o * 32 + r32;
            const uint8_t *ap = buf + L::LR_ACT;
            add_low_rank(o, s, *(const float4_t *)(ap + act_place(row, 4 * k + 2 * h)), *(const float4_t *)(ap + act_place(row, 4 * k + 2 * h + 1)), up);
        }
    };
#pragma unroll
    for (int s = 0; s < LR_AHEAD; s++) {
        if (s >= lr_steps) break;
        add_copied(lds + L::LR, s);
    }
    if constexpr (RANKS) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        for (int c = 0; 2 * c < copied; c++) {
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (2 * c + k >= copied) break;
                add_copied(lds, 2 * c + k);
            }
        }
        __syncthreads();  // (read: the slabs take their place)
    }
    for (int s0 = RANKS ? copied : LFIRST; s0 < nsteps; s0 += LSTEPS) {
        if (RANKS || s0 > LFIRST) load_more(s0);
#pragma unroll
        for (int s = 0; s < LSTEPS; s++)
            if (s0 + s < nsteps) add_step(more[s], s0 + s);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4_t bs = biases(q);
#pragma unroll
        for (int o = 0; o < OWN; o++)
#pragma unroll
            for (int i = 0; i < 4; i++) val[o][4 * q + i] += bs[i];
    }
    if constexpr (NARROW) {
        // the wave's 32 x 32 block through its own slab, in rows of 64 contiguous bytes
        uint16_t *slab = (uint16_t *)(lds + L::SLABS + wave * NARROW_SLAB_BYTES);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            u32x2_t w;
            w[0] = pack_bf16x2(val[0][4 * q], val[0][4 * q + 1]);
            w[1] = pack_bf16x2(val[0][4 * q + 2], val[0][4 * q + 3]);
            *(u32x2_t *)(slab + r32 * NARROW_LD + 8 * q + 4 * h) = w;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the slab is the wave's own, whose LDS operations complete in order)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const int rr = it * 16 + (lane >> 2), cc = (lane & 3) * 8, m = row0 + rr, n = c0 + cc;
            const u32x4_t d = *(const u32x4_t *)(slab + rr * NARROW_LD + cc);
            if (p.out && m < p.M_out && n < p.N_out) __builtin_nontemporal_store(d, (u32x4_t *)(p.out + (size_t)m * p.N_out + n));
        }
        return;
    } else {
    if (rope) {
#pragma unroll
        for (int o = 0; o < MT; o++) {
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 16; e++) ss += val[o][e] * val[o][e];
            ss += __shfl_xor(ss, 32);
            if (h == 0) ssq[(o * 4 + nt) * 32 + r32] = ss;
        }
        // EpilogueRMSNormRope (epilogues.cuh:269-425); the (sin, cos) table is stored in this loop's order, see
        // gemm6_kernel.h
        __syncthreads();
        const uint16_t *nw = (n0 < p.rope_cols / 2 ? p.norm_q : p.norm_k) + nt * 32 + 4 * h;
#pragma unroll
        for (int o = 0; o < MT; o++) {
            int blk = f0 + o;
            blk = blk < (p.rot_rows >> 5) ? blk : (p.rot_rows >> 5) - 1;  // (rows beyond the output are never stored)
            const float4_t *rp = (const float4_t *)p.rotary + ((size_t)blk * 16 + nt * 4) * 64 + lane;
            const float *sp = ssq + o * 128 + r32;
            const float coef = __builtin_amdgcn_rsqf((((sp[0] + sp[32]) + sp[64]) + sp[96]) * (1.0f / 128.0f) + p.norm_eps);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4_t s4 = rp[q * 64];  // sin, cos of two pairs
                const u32x2_t w2 = *(const u32x2_t *)(nw + 8 * q);
#pragma unroll
                for (int pr = 0; pr < 2; pr++) {
                    const float x = val[o][4 * q + 2 * pr] * (coef * bits_f32(w2[pr] << 16));
                    const float y = val[o][4 * q + 2 * pr + 1] * (coef * bits_f32(w2[pr] & 0xFFFF0000u));
                    const float sn = s4[2 * pr], cs = s4[2 * pr + 1];
                    val[o][4 * q + 2 * pr] = x * cs - y * sn;
                    val[o][4 * q + 2 * pr + 1] = x * sn + y * cs;
                }
            }
        }
    }
#pragma unroll
    for (int o = 0; o < MT; o++) {
        if (NEXT && p.silu) {
#pragma unroll
            for (int e = 0; e < 16; e++) val[o][e] *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * val[o][e]));
        }
        if (NEXT && p.gelu) {
#pragma unroll
            for (int e = 0; e < 16; e++) val[o][e] = gelu_tanh(val[o][e]);
        }
        if (NEXT && p.vk && n0 < p.N / 3) {
            // the q third of a linear-attention projection is stored after a ReLU (epilogues.cuh:662-674)
#pragma unroll
            for (int e = 0; e < 16; e++) val[o][e] = __builtin_fmaxf(val[o][e], 0.f);
        }
        uint16_t *slab = (uint16_t *)(lds + o * SLAB_BYTES);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            u32x2_t w;
            w[0] = pack_bf16x2(val[o][4 * q], val[o][4 * q + 1]);
            w[1] = pack_bf16x2(val[o][4 * q + 2], val[o][4 * q + 3]);
            *(u32x2_t *)(slab + r32 * OUT_LD + nt * 32 + 8 * q + 4 * h) = w;
        }
    }
    // the reciprocal smoothing factors of the next layer for the 32 columns a lane quantizes
    float nrs[32];
    const bool quantizes = NEXT && p.qout && wave < 2 * MT;
    if (quantizes) {
        const float4_t *sp = (const float4_t *)(p.next_smooth_rcp + n0 + (lane & 3) * 32);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float4_t v4 = sp[i];
            nrs[4 * i] = v4[0]; nrs[4 * i + 1] = v4[1]; nrs[4 * i + 2] = v4[2]; nrs[4 * i + 3] = v4[3];
        }
    }
    __syncthreads();

    // ---- the bf16 tile, MT slabs of 32 rows, is in LDS ------------------------------------------------------
    if (p.out) {
#pragma unroll
        for (int it = 0; it < MT * 8 / WAVES; it++) {
            const int item = it * WAVES + wave, mt = item >> 3, rr = (item & 7) * 4 + (lane >> 4), cc = (lane & 15) * 8;
            const int m = (f0 + mt) * 32 + rr, n = n0 + cc;
            const u32x4_t d = *(const u32x4_t *)((const uint16_t *)(lds + mt * SLAB_BYTES) + rr * OUT_LD + cc);
            if (m < p.M_out && n < p.N_out) __builtin_nontemporal_store(d, (u32x4_t *)(p.out + (size_t)m * p.N_out + n));
        }
    }
    if (NEXT && p.qkv.q && wave < MT) store_qkv_slab(p.qkv, (const uint16_t *)(lds + wave * SLAB_BYTES), OUT_LD, lane, (f0 + wave) * 32, n0, p.N / 3);
    if (NEXT && p.vk && n0 >= p.N / 3 && wave < MT) {
        VkSums vks;
        litela_clear(vks);
        litela_add_slab(vks, (const uint16_t *)(lds + wave * SLAB_BYTES), OUT_LD, lane);
        const int third = p.N / 3;
        litela_park<true>(vks, p.vk_part + ((size_t)(f0 + wave) * (2 * third / 64) + (n0 - third) / 64) * VK_HEAD_FLOATS, lane);
    }
    if (NEXT && p.next_down) {
        // low-rank down projection of the next layer on the bf16 tile (EpilogueLoraDown, lora.cuh:243-353): the tile's 128
        // columns are one chunk of the next layer's K, whose share goes to the workspace (reduce_shares_kernel in gemm.hip)
        const int RT = p.R_down / 16, r16 = lane & 15, q = lane >> 4;
        for (int item = wave; item < MT * RT * 2; item += WAVES) {
            const int m2 = item & 1, rt = (item >> 1) % RT, mt = (item >> 1) / RT;
            const uint16_t *slab = (const uint16_t *)(lds + mt * SLAB_BYTES);
            float4_t d = {0.f, 0.f, 0.f, 0.f};
            bf16x8_t b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) b[i] = p.next_down[((size_t)(nb * 4 + i) * RT + rt) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const bf16x8_t a = *(const bf16x8_t *)(slab + (16 * m2 + r16) * OUT_LD + 32 * q + 8 * i);
                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[i], d, 0, 0, 0);
            }
            __builtin_nontemporal_store(d, (float4_t *)(p.next_lora_part + (size_t)nb * p.M_pad * p.R_down) + (((size_t)(f0 + mt) * RT + rt) * 2 + m2) * 64 + lane);
        }
    }
    if (quantizes) {
        // EpilogueQuantize (gemm_w4a4.cuh:930-1043): INT4 with the shift and unsigned codes, NVFP4 without
        const int item = (wave & 1) * 64 + lane, rr = item >> 2, qc = item & 3;
        const u32x4_t *sp = (const u32x4_t *)((const uint16_t *)(lds + (wave >> 1) * SLAB_BYTES) + rr * OUT_LD + qc * 32);
        float y[32];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const u32x4_t v4 = sp[i];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float lo = bits_f32(v4[j] << 16), hi = bits_f32(v4[j] & 0xFFFF0000u);
                if (!FP4) {
                    lo = round_to_bf16(__fadd_rn(lo, 0.171875f));
                    hi = round_to_bf16(__fadd_rn(hi, 0.171875f));
                }
                y[8 * i + 2 * j] = smooth_quotient(lo, nrs[8 * i + 2 * j]);
                y[8 * i + 2 * j + 1] = smooth_quotient(hi, nrs[8 * i + 2 * j + 1]);
            }
        }
        const int m = (f0 + (wave >> 1)) * 32 + rr, gidx = (n0 + qc * 32) / 64, ngroups_out = p.N / 64;
        if constexpr (!FP4) {
            u32x4_t lo4;
            u32x2_t hi2;
            float sc;
            quantize_int4_half_group_e2m3<true>(y, 1, lo4, hi2, sc);
            if ((qc & 1) == 0) ((uint16_t *)p.oscales)[(size_t)gidx * p.M_pad + m] = (uint16_t)f32_to_bf16_bits(sc);
            uint8_t *frag = p.qout + (((size_t)(m / ACT_BLOCK_ROWS) * ngroups_out + gidx) * 4 + (m % ACT_BLOCK_ROWS) / 32) * FRAG_BYTES;
            const int slot = (m % 32) + 32 * (qc & 1);
            *(u32x4_t *)(frag + slot * 16) = lo4;
            *(u32x2_t *)(frag + 1024 + slot * 8) = hi2;
        } else {
            u32x4_t words;
            uint32_t sc[2];
            quantize_nvfp4_two_groups(y, words, sc);
            ((uint16_t *)p.oscales)[((size_t)gidx * p.M_pad + m) * 2 + (qc & 1)] = (uint16_t)(sc[0] | (sc[1] << 8));  // [N/64][M_pad][4]
            *(u32x4_t *)(p.qout + ((size_t)(m / 32) * ngroups_out + gidx) * TILE_BYTES + (m % 32) * 32 + 16 * (qc & 1)) = words;
        }
    }
    }
}

template <bool FP4, int MT, int NT, int WN, int KP, int DEPTH, bool NEXT, bool RANKS>
__global__ void __launch_bounds__(64 * WN * KP, WN == 4 ? 3 : 2) gemm_direct_kernel(GemmParams p) {
    if constexpr (two_heights(FP4, MT, NT * WN)) {
        const int full = p.full_blocks * (p.N / (32 * NT * WN)), block = (int)blockIdx.x;
        if (block < full) {
            const int v = tile_of(block, full), nb = v / p.full_blocks;
            output_tile<FP4, 2, NT, WN, KP, DEPTH, NEXT, RANKS>(p, nb, (v - nb * p.full_blocks) * 2);
        } else {
            // (as deep a ring as the launches of 32-row tiles alone have)
            const int half_blocks = p.row_blocks - p.full_blocks, v = tile_of(block - full, (int)gridDim.x - full), nb = v / half_blocks;
            output_tile<FP4, 1, NT, WN, KP, FP4_RING<1>, NEXT, RANKS>(p, nb, p.full_blocks * 2 + v - nb * half_blocks);
        }
    } else {
        const int v = tile_of((int)blockIdx.x, (int)gridDim.x), nb = v / p.row_blocks;
        output_tile<FP4, MT, NT, WN, KP, DEPTH, NEXT, RANKS>(p, nb, (v - nb * p.row_blocks) * MT);
    }
}

template <bool FP4, int MT, int NT, int WN, int KP, int DEPTH, bool NEXT, bool RANKS = false>
int launch_direct(const GemmParams &params, hipStream_t stream) {
    auto kern = gemm_direct_kernel<FP4, MT, NT, WN, KP, DEPTH, NEXT, RANKS>;
    using L = Lds<MT, NT, WN, KP, DEPTH>;
    static bool lds_reserved[64] = {false};  // set once per device (racing first calls both set it, which is harmless)
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return fail(SVDQ_ELAUNCH, "gemm: cannot identify the current device");
    if (!lds_reserved[dev]) {
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, L::bytes(L::LR_AHEAD));
        if (e != hipSuccess) return fail(SVDQ_ELAUNCH, "gemm: cannot reserve %d bytes of LDS: %s", L::bytes(L::LR_AHEAD), hipGetErrorString(e));
        lds_reserved[dev] = true;
    }
    GemmParams p = params;
    const int tiles = p.row_blocks * (p.N / (32 * NT * WN));
    p.lr_steps = L::lr_steps(p.R_up, tiles > 2 * compute_units(dev));
    SVDQ_LAUNCH(kern, dim3((unsigned)tiles), dim3(64 * WN * KP), L::bytes(p.lr_steps), stream, p);
    return check_launch("gemm_w4a4 (few rows)");
}

// NVFP4, tiles of 32 (shape 1) or 64 rows x 128 columns
template <bool NEXT, bool RANKS>
int launch_fp4(const GemmParams &p, int shape, hipStream_t stream) {
    if (shape == 1) return launch_direct<true, 1, 4, 1, 4, FP4_RING<1>, NEXT, RANKS>(p, stream);
    return launch_direct<true, 2, 4, 1, 4, FP4_RING<2>, NEXT, RANKS>(p, stream);
}

}  // namespace direct
}  // namespace svdq
