// Entry points of the library that only this package's own host code calls: not part of the C ABI.
#pragma once

#include "../../include/svdq_amd.h"

#ifdef __cplusplus
extern "C" {
#endif

// svdq_gemm_w4a4 (or, with `noalloc`, svdq_gemm_w4a4_noalloc) of a call that writes no `out` and whose caller reads only the first
// `rows` rows of qout / oscales / next_lora_act_out: what the other rows hold afterwards is unspecified.  The fused MLP's
// first GEMM: M = 1157 of 1280 padded rows.
int svdq_gemm_w4a4_rows(const svdq_gemm_args *args, int64_t rows, int noalloc, void *stream);

// Which kernel a GEMM call takes and how it divides the work (zero where a field does not apply).
typedef struct svdq_gemm_plan {
    int32_t few_rows;      // 0: a kernel with large tiles; 1, 2: the few-rows kernel in tiles of 32, 64 rows,
    int32_t row_blocks;    // so many along M (64-row blocks of the rows, where 32-row ones take the place of some: full_blocks, low_blocks)
    int32_t full_blocks;   // INT4, large tiles: row blocks of 128 rows (NVFP4, few rows, 64 x 128: of 64 rows),
    int32_t half_blocks;   // of 64 rows behind them,
    int32_t kparts;        // and parts along K of every tile
    int32_t workgroups;    // NVFP4, large tiles: persistent workgroups;
    int32_t shared_tiles;  // some tiles are shared by two or more of them
    int32_t columns;       // few rows: columns of a tile (32, 64 or 128),
    int32_t shared_rows;   // its waves split the columns and share the rows' operands through LDS;
    int32_t copied_ranks;  // the low-rank operands come through LDS (NVFP4, tiles of 128 columns);
    int32_t low_blocks;    // NVFP4, 64 x 128: row blocks of 32 rows behind the full ones
} svdq_gemm_plan;

// What svdq_gemm_w4a4 (`rows` > 0: svdq_gemm_w4a4_rows) would do with these arguments on a GPU of so many compute units.  Checks the
// arguments as the call does, launches nothing and needs no GPU.
int svdq_gemm_plan_of(const svdq_gemm_args *args, int64_t rows, int compute_units, svdq_gemm_plan *plan);

// The work of workgroup `block` of an INT4 launch with large tiles.
typedef struct svdq_gemm_tile {
    int32_t row, rows;     // first row, height
    int32_t column_block;  // of 256 columns
    int32_t part;          // along K
    int32_t row_block;     // its number among the blocks of both heights
    int32_t tile;          // the number that the parts of a tile meet under
} svdq_gemm_tile;
void svdq_gemm_int4_tile(const svdq_gemm_plan *plan, int64_t N, int block, svdq_gemm_tile *tile);
// The same of a few-rows launch (column_block: of plan->columns; part 0, tile its number down the rows first); returns the number of workgroups.
int svdq_gemm_few_rows_tile(const svdq_gemm_plan *plan, int64_t N, int block, svdq_gemm_tile *tile);

// The asynchronous copies of the low-rank operands in tiles of 64 x 128 whose waves share the rows (`form` 0) and in tiles of 32 (1) and 64 rows (2) of copied_ranks.
typedef struct svdq_gemm_low_rank {
    int32_t first, end;       // LDS that may hold them, in bytes: what the launch has (form 0, three workgroups per compute unit or two), the place of the sums
    int32_t steps;            // 16-rank steps that come this way
    int32_t chunk, act;       // bytes of 32 ranks; where in them lora_act's stand
    int32_t up_requests, act_requests;  // a KB each, 64 lanes of 16 bytes, of 32 ranks
} svdq_gemm_low_rank;
void svdq_gemm_low_rank_of(int form, int rank, int three, svdq_gemm_low_rank *copies);
// Byte offsets of what lane `lane` of request `request` of chunk `chunk` reads, from the operand's first column (`act`: row) of the tile, which is `first`, on
int64_t svdq_gemm_low_rank_copied(int act, int first, int rank, int chunk, int request, int lane);
// and of 16-byte piece `piece` of a column's (row's) 32 ranks in LDS, from the chunk's lora_up (lora_act) on.
int svdq_gemm_low_rank_place(int act, int index, int piece);

#ifdef __cplusplus
}
#endif
