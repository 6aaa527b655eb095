// The few-rows GEMM with tiles narrower than 128 columns (plain epilogue, either precision): -DSVDQ_VARIANT=0 tiles as wide as high,
// 1 the others; two translation units that build in parallel.
#include "gemm_direct_kernel.h"
#include "internal_api.h"

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

#if SVDQ_VARIANT == 0
// The host's model of the low-rank operands' copies asks the kernel's own functions and layouts.
using Shared = svdq::direct::Lds<2, 1, 4, 1, 3>;
extern "C" void svdq_gemm_low_rank_of(int form, int rank, int three, svdq_gemm_low_rank *copies) {
    using namespace svdq::direct;
    if (form == 0) {
        const int steps = Shared::lr_steps(rank, three != 0);
        *copies = svdq_gemm_low_rank{Shared::LR, Shared::bytes(steps), steps, Shared::LR_CHUNK, Shared::LR_ACT, 8, 8};
        return;
    }
    auto ranks = [&](auto layout, int mt) {
        using L = decltype(layout);
        const int most = 2 * (L::SUMS / L::LR_CHUNK), steps = rank / 16 < most ? rank / 16 : most;
        *copies = svdq_gemm_low_rank{0, L::SUMS, steps, L::LR_CHUNK, L::LR_ACT, 8, 4 * mt};
    };
    if (form == 1) ranks(Lds<1, 4, 1, 4, FP4_RING<1>>{}, 1);
    else ranks(Lds<2, 4, 1, 4, FP4_RING<2>>{}, 2);
}
extern "C" int64_t svdq_gemm_low_rank_copied(int act, int first, int rank, int chunk, int request, int lane) {
    using namespace svdq::direct;
    const bool half = rank / 16 - 2 * chunk < 2;
    return act ? (int64_t)act_base(first, rank, chunk) + act_copied(request, lane, rank, half) : (int64_t)up_base(first, rank, chunk) + up_copied(request, lane, rank, half);
}
extern "C" int svdq_gemm_low_rank_place(int act, int index, int piece) { return act ? svdq::direct::act_place(index, piece) : svdq::direct::up_place(index, piece); }
#endif
