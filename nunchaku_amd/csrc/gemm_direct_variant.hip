// One translation unit per variant of the few-rows GEMM (compiled with -DSVDQ_VARIANT=0: INT4, plain epilogue, 1: INT4
// with the next-layer / norm + rotary / SiLU epilogue, 2 and 3: the same for NVFP4) so that they build in parallel.
#include "gemm_direct_kernel.h"

namespace svdq {
namespace direct {

#if SVDQ_VARIANT == 0
#define SVDQ_NAME launch_int4_plain
#elif SVDQ_VARIANT == 1
#define SVDQ_NAME launch_int4_next
#elif SVDQ_VARIANT == 2
#define SVDQ_NAME launch_fp4_plain
#else
#define SVDQ_NAME launch_fp4_next
#endif

int SVDQ_NAME(const GemmParams &p, int shape, hipStream_t stream) {
    constexpr bool NEXT = SVDQ_VARIANT & 1;
#if SVDQ_VARIANT >= 2
    return launch_fp4<NEXT, false>(p, shape, stream);
#else
    // (the ring of k-groups on their way as deep as the registers of two waves per SIMD allow)
    if (shape == 1) return launch_direct<false, 1, 4, 1, 4, 1, NEXT>(p, stream);
    return launch_direct<false, 2, 2, 2, 2, 1, NEXT>(p, stream);
#endif
}

}  // namespace direct
}  // namespace svdq
