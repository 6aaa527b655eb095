// The NVFP4 few-rows GEMM of ranks above 32 in tiles of 128 columns (compiled with -DSVDQ_VARIANT=0: plain epilogue, 1: the others): two translation
// units that build in parallel.
#include "gemm_direct_kernel.h"

namespace svdq {
namespace direct {

#if SVDQ_VARIANT == 0
int launch_fp4_ranks_plain(const GemmParams &p, int shape, hipStream_t stream) {
#else
int launch_fp4_ranks_next(const GemmParams &p, int shape, hipStream_t stream) {
#endif
    return launch_fp4<SVDQ_VARIANT != 0, true>(p, shape, stream);
}

}  // namespace direct
}  // namespace svdq
