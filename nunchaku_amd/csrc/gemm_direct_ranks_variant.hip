// The NVFP4 few-rows GEMM of ranks above 32 in tiles of 128 columns (compiled with -DSVDQ_VARIANT=0: plain epilogue, 1: the others): two translation
// units that build in parallel.  Tiles and rings are those of gemm_direct_variant.hip.
#include "gemm_direct_kernel.h"

namespace svdq {
namespace direct {

#if SVDQ_VARIANT == 0
int launch_fp4_ranks_plain(const GemmParams &p, int shape, hipStream_t stream) {
#else
int launch_fp4_ranks_next(const GemmParams &p, int shape, hipStream_t stream) {
#endif
    constexpr bool NEXT = SVDQ_VARIANT;
    if (shape == 1) return launch_direct<true, 1, 4, 1, 4, 2, NEXT, true>(p, stream);
    return launch_direct<true, 2, 4, 1, 4, 1, NEXT, true>(p, stream);
}

}  // namespace direct
}  // namespace svdq
