// The few-rows GEMM with tiles narrower than 128 columns (plain epilogue, either precision): -DSVDQ_VARIANT=0 tiles as wide as high,
// 1 the others; two translation units that build in parallel.
#include "gemm_direct_kernel.h"

namespace svdq {
namespace direct {

#if SVDQ_VARIANT == 0
#define SVDQ_NAME launch_square
#else
#define SVDQ_NAME launch_oblong
#endif

// Tiles of 32 mt rows x 32 nt columns.  (k-groups on their way: of 32 x 32 tiles a third one gave nothing more, M = 16 ... 512, K = 1024 ... 12288.)
template <bool FP4>
int launch_narrow(const GemmParams &p, int mt, hipStream_t stream) {
#if SVDQ_VARIANT == 0
    return mt == 1 ? launch_direct<FP4, 1, 1, 1, 4, 2, false>(p, stream) : launch_direct<FP4, 2, 2, 1, 4, FP4 ? 2 : 1, false>(p, stream);
#else
    return mt == 1 ? launch_direct<FP4, 1, 2, 1, 4, 2, false>(p, stream) : launch_direct<FP4, 2, 1, 1, 4, 2, false>(p, stream);
#endif
}

// INT4, tiles of 64 rows x 128 columns whose waves split the columns only: plain epilogue (0), the others (1)
#if SVDQ_VARIANT == 0
int launch_staged_plain(const GemmParams &p, hipStream_t stream) { return launch_direct<false, 2, 1, 4, 1, 3, false>(p, stream); }
#else
int launch_staged_next(const GemmParams &p, hipStream_t stream) { return launch_direct<false, 2, 1, 4, 1, 3, true>(p, stream); }
#endif

int SVDQ_NAME(const GemmParams &p, bool fp4, int mt, hipStream_t stream) { return fp4 ? launch_narrow<true>(p, mt, stream) : launch_narrow<false>(p, mt, stream); }

}  // namespace direct
}  // namespace svdq
