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

#ifdef __cplusplus
}
#endif
