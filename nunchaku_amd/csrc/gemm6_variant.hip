// One translation unit per variant of the INT4 GEMM (compiled with -DSVDQ_VARIANT=0: plain epilogue,
// 1: with the next-layer / norm + rotary / SiLU epilogue, 2 and 3: the same without the unrolled main loop of the 128-row tiles) so
// that they build in parallel.
#include "gemm6_kernel.h"

namespace svdq {
namespace g6 {

#if SVDQ_VARIANT == 0
int launch_plain(const Params &p, int nwg, hipStream_t stream) { return launch_gemm6<false, true>(p, nwg, stream); }
#elif SVDQ_VARIANT == 1
int launch_next(const Params &p, int nwg, hipStream_t stream) { return launch_gemm6<true, true>(p, nwg, stream); }
#elif SVDQ_VARIANT == 2
int launch_plain_rolled(const Params &p, int nwg, hipStream_t stream) { return launch_gemm6<false, false>(p, nwg, stream); }
#else
int launch_next_rolled(const Params &p, int nwg, hipStream_t stream) { return launch_gemm6<true, false>(p, nwg, stream); }
#endif

}  // namespace g6
}  // namespace svdq
