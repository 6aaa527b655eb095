// Host entry point of operator 2 (argument validation, kernel variant selection).  The device code
// lives in gemm_kernel.h and is instantiated per variant in gemm_variant.hip.
#include "gemm_params.h"
#include "internal_api.h"

using namespace svdq;

namespace svdq {
int launch_gemm_fp4_v4(const GemmParams &p, int nwg, hipStream_t stream);
int launch_gemm_fp4_v5(const GemmParams &p, int nwg, hipStream_t stream);
namespace direct {
int launch_int4_plain(const GemmParams &p, int shape, hipStream_t stream);
int launch_int4_next(const GemmParams &p, int shape, hipStream_t stream);
int launch_fp4_plain(const GemmParams &p, int shape, hipStream_t stream);
int launch_fp4_next(const GemmParams &p, int shape, hipStream_t stream);
int launch_fp4_ranks_plain(const GemmParams &p, int shape, hipStream_t stream);
int launch_fp4_ranks_next(const GemmParams &p, int shape, hipStream_t stream);
int launch_square(const GemmParams &p, bool fp4, int mt, hipStream_t stream);
int launch_oblong(const GemmParams &p, bool fp4, int mt, hipStream_t stream);
int launch_staged_plain(const GemmParams &p, hipStream_t stream);
int launch_staged_next(const GemmParams &p, hipStream_t stream);
}  // namespace direct
namespace g6 {
int launch_plain(const Params &p, int nwg, hipStream_t stream);
int launch_next(const Params &p, int nwg, hipStream_t stream);
}  // namespace g6
}  // namespace svdq

#include <math.h>
#include <mutex>
#include <stdlib.h>
#include <vector>

namespace {
// Workspace of one (device, stream) pair: launches on one stream run one after the other and can share
// it, launches on different streams may overlap and must not.  It is allocated the first time a launch
// needs one.  A block that has been handed to a launch is never freed behind the caller's back: a HIP graph
// captured through this entry point holds the block's address for as long as the graph lives.  A pair
// that needs more than it has gets a new, larger block (at least half as large again, so that all the
// blocks a pair ever outgrew stay below twice its present one) and the old one is retired, still
// allocated; svdq_release_workspaces is the only place that frees.  The first `zero_bytes` hold arrival
// counters: zero when allocated, and every launch that completes leaves them at zero again.  The rest is
// scratch (parked partial sums, low-rank shares).
struct Workspace {
    int dev;
    hipStream_t stream;
    uint8_t *ptr;
    size_t zero_bytes, scratch_bytes;
    bool dirty;  // a launch failed: the zero region is cleared again before the next use
};
struct Retired {
    int dev;
    void *ptr;
};
std::vector<Workspace> g_ws;
std::vector<Retired> g_retired;
std::mutex g_ws_mutex;  // held from the look-up until the launch that uses the workspace has been enqueued

__global__ void zero_f32_kernel(float *p, int64_t n) {
    const int64_t i = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) * 4;
    if (i + 3 < n) *(float4_t *)(p + i) = float4_t{0.f, 0.f, 0.f, 0.f};
    else for (int64_t j = i; j < n; j++) p[j] = 0.f;
}

// The sum of float4 number `item` over n shares that lie `stride` float4 apart, worked out by the PARTS threads of a
// workgroup that have the same threadIdx.x % 32: each adds a PARTS-th of the shares in ascending order, eight requests in
// flight, and the first of them adds the parts in ascending order.  `item` of the threads without work is any valid one.
// Valid in the workgroup's first 32 threads.
template <int PARTS>
__device__ inline float4_t sum_of_shares(const float4_t *part, size_t item, size_t stride, int n) {
    __shared__ float4_t parts[PARTS][32];
    const int e = threadIdx.x >> 5, lane = threadIdx.x & 31;
    const int first = n * e / PARTS, last = n * (e + 1) / PARTS;
    float4_t sum = float4_t{0.f, 0.f, 0.f, 0.f};
    for (int b0 = first; b0 < last; b0 += 8) {
        float4_t v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = part[(size_t)(b0 + u < last ? b0 + u : last - 1) * stride + item];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (b0 + u < last) sum += v[u];
    }
    parts[e][lane] = sum;
    __syncthreads();
    if (e == 0) {
#pragma unroll
        for (int u = 1; u < PARTS; u++) sum += parts[u][lane];
    }
    return sum;
}

// Sums the shares that the column blocks (INT4 kernel: 256 columns each) or chunks (NVFP4 and few-rows kernels: 128 columns)
// of a GEMM launch left for the next layer's low-rank projection, and writes lora_act [M_pad][R] row-major.  A share is
// [M_pad / 32 slabs][R / 16 rank tiles][2 halves of 16 rows][64 lanes] x float4, lane l holding rows 4 (l / 16) + [0, 4),
// rank l % 16 of a 16 x 16 tile (the result registers of the matrix instruction).
// Bound by latency at few rows, where one thread per sum had 6 to 12 rounds of requests to wait for: 96 shares of 1280 rows, rank
// 32, 11.5 us before and 5.5 now; 48 shares of 4608 rows (28 MB) 6.2 and 6.2.
template <int PARTS>
__global__ void __launch_bounds__(32 * PARTS) reduce_shares_kernel(const float4_t *part, float *out, int nshares, int M_pad, int R) {
    const int RT = R / 16, quads = M_pad * R / 4;  // (M_pad is a multiple of 256 and R of 16: whole workgroups)
    const int item = blockIdx.x * 32 + (threadIdx.x & 31);
    const float4_t sum = sum_of_shares<PARTS>(part, item, quads, nshares);
    if (threadIdx.x >= 32) return;
    const int ln = item & 63, m2 = (item >> 6) & 1, rest = item >> 7;  // rest = slab * RT + rank tile
    const int rt = rest % RT, slab32 = rest / RT;
    const int row = slab32 * 32 + 16 * m2 + 4 * (ln >> 4), rank = 16 * rt + (ln & 15);
#pragma unroll
    for (int e = 0; e < 4; e++) out[(size_t)(row + e) * R + rank] = sum[e];
}

// Sums the linear-attention shares of the row blocks of a GEMM launch (gemm_params.h; per row block and head 1056 floats:
// the 32 x 32 part [i][j] in the order of the matrix instruction's result registers, element e of lane l at
// ((e / 4) * 64 + l) * 4 + e % 4 with i = 8 (e / 4) + 4 (l / 32) + e % 4, j = l % 32; then the 32 column sums) into
// out_vk [batch][head][33][32].  A workgroup's 32 float4 are 4 rows i of all 32 columns j, or the 8 of the column sums.
// The shares are those of row blocks of vk_block rows up to row `full_rows` and of 64 rows from there on; a batch entry is
// vk_rows of them.
template <int PARTS>
__global__ void __launch_bounds__(32 * PARTS) reduce_vk_kernel(const float4_t *part, float *out, int vk_rows, int vk_block, int full_rows, int heads) {
    constexpr int QUADS = VK_HEAD_FLOATS / 4, PIECES = (QUADS + 31) / 32;
    const int piece = blockIdx.x % PIECES, head = (blockIdx.x / PIECES) % heads, b = blockIdx.x / (PIECES * heads);
    const int lane = threadIdx.x & 31, quad = piece * 32 + lane;
    auto slots_before = [&](int row) { return row <= full_rows ? row / vk_block : full_rows / vk_block + (row - full_rows) / 64; };
    const int slot = slots_before(b * vk_rows);
    const size_t item = ((size_t)slot * heads + head) * QUADS + (quad < QUADS ? quad : QUADS - 1);
    const float4_t sum = sum_of_shares<PARTS>(part, item, (size_t)heads * QUADS, slots_before((b + 1) * vk_rows) - slot);
    if (threadIdx.x >= 32 || quad >= QUADS) return;
    float *o = out + ((size_t)b * heads + head) * VK_HEAD_FLOATS;
    if (piece == PIECES - 1) {
        *(float4_t *)(o + 1024 + 4 * lane) = sum;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) o[(4 * piece + e) * 32 + lane] = sum[e];  // (pieces 2 g and 2 g + 1 are lanes 0-31 and 32-63 of group g)
}
static_assert(VK_HEAD_FLOATS == 33 * 32, "eight whole pieces of the 32 x 32 part, then the column sums");

void clear_zero_region(Workspace *w) {
    const int64_t n = (int64_t)(w->zero_bytes / 4);
    if (n > 0) SVDQ_LAUNCH(zero_f32_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, w->stream, (float *)w->ptr, n);
    w->dirty = false;
}

// (the caller holds g_ws_mutex) returns nullptr, with the error text set, on failure
Workspace *get_workspace(int dev, hipStream_t stream, size_t zero_bytes, size_t scratch_bytes) {
    Workspace *w = nullptr;
    for (Workspace &cand : g_ws)
        if (cand.dev == dev && cand.stream == stream) w = &cand;
    if (w && w->zero_bytes >= zero_bytes && w->scratch_bytes >= scratch_bytes) {
        if (w->dirty) clear_zero_region(w);
        return w;
    }
    // A new block is needed.  Not while the stream is being captured: the allocation is not a stream
    // operation, and the runtime refuses it in a capture of the global mode.
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) == hipSuccess && capturing != hipStreamCaptureStatusNone) {
        fail(SVDQ_EUNSUPPORTED, "gemm: this call needs %zu bytes of workspace that the stream's pair does not have yet, and the stream is being "
             "captured: make the call once before the capture, or use svdq_gemm_w4a4_noalloc", zero_bytes + scratch_bytes);
        return nullptr;
    }
    if (w) {
        if (zero_bytes < w->zero_bytes) zero_bytes = w->zero_bytes;
        if (scratch_bytes < w->scratch_bytes + w->scratch_bytes / 2) scratch_bytes = w->scratch_bytes + w->scratch_bytes / 2;
    }
    zero_bytes = (zero_bytes + (1u << 20) - 1) & ~(size_t)((1u << 20) - 1);  // in steps of 1 MB: few regrows
    uint8_t *ptr = nullptr;
    hipError_t e = hipMalloc((void **)&ptr, zero_bytes + scratch_bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        fail(SVDQ_ELAUNCH, "gemm: cannot allocate %zu bytes of workspace: %s", zero_bytes + scratch_bytes, hipGetErrorString(e));
        return nullptr;
    }
    if (w) {
        // launches already enqueued on this stream (and graphs that captured this block) go on using the old block
        g_retired.push_back(Retired{dev, w->ptr});
    } else {
        g_ws.push_back(Workspace{dev, stream, nullptr, 0, 0, false});
        w = &g_ws.back();
    }
    w->ptr = ptr;
    w->zero_bytes = zero_bytes;
    w->scratch_bytes = scratch_bytes;
    clear_zero_region(w);  // on the caller's stream: ordered before the launch that follows
    return w;
}

// ---- the scratch of svdq_gemm_w4a4_noalloc --------------------------------------------------------
// A fixed array in device memory, one copy per GPU, held until the process ends: first the region that
// must be zero when a launch starts (arrival counters), then parked partial sums and low-rank shares.
constexpr size_t NOALLOC_ZERO_BYTES = 1u << 20, NOALLOC_SCRATCH_BYTES = 80u << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_ZERO_BYTES + NOALLOC_SCRATCH_BYTES];
uint8_t *g_scratch_ptr[64] = {nullptr};  // the array's device address on each GPU, asked once per GPU
// Held from before the fill kernel until the last kernel of a call that uses the array has been enqueued: between the GEMM and
// the sums of its shares no other thread's GEMM on the stream may write shares of its own to the same place.
std::mutex g_scratch_mutex;

// (the caller holds g_scratch_mutex) the array's address on device `dev` (which is the current device), or nullptr with the error
// text set
uint8_t *scratch_address(int dev) {
    if (dev < 0 || dev >= 64) {
        fail(SVDQ_ELAUNCH, "gemm: device index %d out of range", dev);
        return nullptr;
    }
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            fail(SVDQ_ELAUNCH, "gemm: cannot locate the scratch array on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        g_scratch_ptr[dev] = (uint8_t *)ptr;
    }
    return g_scratch_ptr[dev];
}

// Where a launch gets its workspace from: the per-(device, stream) allocation of svdq_gemm_w4a4, or the
// fixed scratch array of svdq_gemm_w4a4_noalloc.
struct WorkspaceView {
    uint8_t *zero;     // zero_bytes that are zero when the launch starts
    uint8_t *scratch;  // scratch_bytes of anything
    Workspace *owner;  // the allocation behind it (nullptr for the fixed array)
};

// Every call that uses a workspace holds this lock from here until all its launches have been enqueued.
std::mutex &workspace_mutex(bool noalloc) { return noalloc ? g_scratch_mutex : g_ws_mutex; }

// (the caller holds workspace_mutex(noalloc)) false, with the error text set, on failure
bool acquire_workspace(bool noalloc, int dev, hipStream_t st, size_t zero_bytes, size_t scratch_bytes, WorkspaceView *v) {
    if (!noalloc) {
        Workspace *w = get_workspace(dev, st, zero_bytes, scratch_bytes);
        if (!w) return false;
        *v = WorkspaceView{w->ptr, w->ptr + w->zero_bytes, w};
        return true;
    }
    if (zero_bytes > NOALLOC_ZERO_BYTES || scratch_bytes > NOALLOC_SCRATCH_BYTES) {
        fail(SVDQ_EUNSUPPORTED, "gemm (noalloc): this call needs %zu + %zu bytes of workspace, the fixed scratch holds %zu + %zu; use svdq_gemm_w4a4",
             zero_bytes, scratch_bytes, NOALLOC_ZERO_BYTES, NOALLOC_SCRATCH_BYTES);
        return false;
    }
    uint8_t *base = scratch_address(dev);
    if (!base) return false;
    // The array keeps the last call's contents.  A launch that completes leaves its counters and sums at
    // zero, one that failed or was aborted does not: what this launch needs to be zero is cleared (by a
    // fill kernel, which a caller's graph capture can record).
    const int64_t n = (int64_t)((zero_bytes + 15) / 16 * 4);
    if (n > 0) SVDQ_LAUNCH(zero_f32_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, st, (float *)base, n);
    *v = WorkspaceView{base, base + NOALLOC_ZERO_BYTES, nullptr};
    return true;
}

// The small kernels behind a GEMM that left shares in the workspace: the shares of the next layer's low-rank projection
// (one per column block) and the linear-attention sums (one per vk_block rows, from row `full_rows` on one per 64), each
// added in ascending order.
template <typename P>
int add_shares(const P &p, int rows, int nshares, int vk_block, int full_rows, hipStream_t st) {
    if (p.next_down) {
        const int quads = (rows + 31) / 32 * 32 * p.R_down / 4;
        auto launch = [&](auto PARTS) {
            constexpr int parts = decltype(PARTS)::value;
            SVDQ_LAUNCH(reduce_shares_kernel<parts>, dim3((unsigned)(quads / 32)), dim3(32 * parts), 0, st, (const float4_t *)p.next_lora_part, p.next_lora_out, nshares,
                        p.M_pad, p.R_down);
        };
        if (nshares <= 32) launch(std::integral_constant<int, 4>{});
        else if (nshares <= 64) launch(std::integral_constant<int, 8>{});
        else launch(std::integral_constant<int, 16>{});
        const int rc = check_launch("gemm_w4a4 (low-rank shares)");
        if (rc != SVDQ_OK) return rc;
    }
    if (p.vk) {
        const int heads = p.N / 96, batch = p.M_pad / p.vk_rows;
        auto launch = [&](auto PARTS) {
            constexpr int parts = decltype(PARTS)::value;
            SVDQ_LAUNCH(reduce_vk_kernel<parts>, dim3((unsigned)(batch * heads * 9)), dim3(32 * parts), 0, st, (const float4_t *)p.vk_part, p.vk, p.vk_rows, vk_block, full_rows,
                        heads);
        };
        if (p.vk_rows <= 1024) launch(std::integral_constant<int, 4>{});
        else launch(std::integral_constant<int, 8>{});
        return check_launch("gemm_w4a4 (linear-attention sums)");
    }
    return SVDQ_OK;
}

// Into how many parts along K the tiles of an INT4 launch are split when the caller leaves that to the library.
// Launches with more tiles than compute units are not split: every part parks 128 KB of sums and the last one fetches
// them all, which only pays while compute units would otherwise stand idle.  Below that, a model of the time in us,
// fitted to launches of 24 ... 216 tiles at K = 3072 and 12288 on 256 compute units: a k-group takes a workgroup 0.55 us
// while it has its compute unit to itself and 0.95 us when two share one; prologue and epilogue 4.4; a split costs
// 5.3 + 2.6 per part beyond the first (four parts, whose last one keeps its own sums in registers: 11.5), half as much
// again when compute units are shared.  Measured, whole / best split: 24 tiles at K = 3072 31.2 / 22.5 (4 parts; 3
// parts 24.2), 72 tiles 31.3 / 27.3 (3), 96 tiles 31.8 / 31.0 (2; not split), 144 tiles 32.1 / 38.1 (not split);
// K = 12288: 24 tiles 105.9 / 39.6 (6), 72 tiles 105.6 / 51.7 (3), 144 tiles 106.2 / 78.4 (3).  (The price of a split is that of requests made lane by lane;
// since they have scalar descriptors it is up to 1.4 us less, M = 856, K = 4992, N = 2432 in three parts 30.7 -> 29.5.)
// `time`: the model's time in us for the choice where there is one.
int choose_kparts(int ntiles, int kgroups, int ncu, double *time) {
    *time = 0.0;
    if (ntiles > ncu) return 1;
    int best = 1;
    double best_t = 0.55 * kgroups + 4.4;
    for (int k : {2, 3, 4, 6, 8}) {
        const int units = ntiles * k, g = (kgroups + k - 1) / k;
        if (g < 12 || units > 2 * ncu) break;
        const bool shared = units > ncu;
        const double t = g * (shared ? 0.95 : 0.55) + 4.4 + (k == 4 ? 11.5 : 5.3 + 2.6 * (k - 1)) * (shared ? 1.5 : 1.0);
        if (t < (best == 1 ? 0.90 : 0.95) * best_t) {  // a split has to pay clearly; more parts likewise
            best = k;
            best_t = t;
        }
    }
    *time = best_t;
    return best;
}

// (the kernels with the next-layer epilogue also carry the norm + rotary, SiLU and linear-attention epilogues)
bool needs_next_epilogue(const svdq_gemm_args *a) {
    return a->qout != nullptr || a->next_lora_down != nullptr || a->rotary_emb != nullptr || a->fuse_silu || a->out_vk != nullptr;
}

// Rows the call has to work out: those of `out` where nothing else is written, those that svdq_gemm_w4a4_rows names where
// `out` is not given, all of them otherwise.
int rows_needed(const svdq_gemm_args *a) {
    if (a->out_q || a->out_vk || (a->out && (a->qout || a->next_lora_down)) || a->M_out == 0) return (int)a->M_pad;
    return (int)a->M_out;
}

// How the rows of an INT4 launch are divided into blocks of 128 rows, and blocks of 64 rows behind them, when the caller
// leaves the split along K to the library.  The last tiles of a launch leave compute units idle for the time of a whole
// tile (the hardware hands tiles to the emptiest compute unit; with 1296 tiles 16 of 256 work 22 us longer than the
// others); in tiles of half the height the last rows fill them up.
// A model of the busiest compute unit's time, in units of a whole tile alone on one, fitted to every division considered of 700
// shapes (M = 256 ... 18432, K = 1024 ... 12288, N = 1024 ... 21504) and checked on 700 others: a pair of whole tiles side by side
// takes 1.55, of half tiles 0.9, a half tile alone 0.7; a half tile next to a last odd whole one 1.2 together with it, two of them 2.0
// (the second starts when the first is done), each one more 0.45.
// Every compute unit gets `tiles / ncu` whole tiles or one more, the half tiles go where they end first.  Considered are whole
// tiles only, whole tiles up to the last and the last but one multiple of the compute units, and (few tiles) half tiles only; a
// division with half tiles has to be 4 % faster by the model.  Measured, whole tiles / the choice: M = 4608, K = 3072, N = 9216
// 140 / 131 us; M = 4096, K = 2304, N = 6912 72.3 / 66.3; M = 1024, K = 3072, N = 9216 44.5 / 34.3; M = 505 of the same layer 32.9 / 28.7
// (with the main loop in whole turns of its ring 122, and 25.3 at M = 505).
// Over the 700 other shapes 1.10 times as fast as whole tiles, 0.2 % off the best division measured, more than 3 % slower than whole
// tiles in one.  (With 1.1 and 0.25, where three half tiles fit behind an odd whole one: slower in six, M = 4096, K = 3072, N = 9216, which
// is whole tiles only now, 129 against 124.)
double half_tiles_time(int n) { return 0.9 * (n / 2) + 0.7 * (n % 2); }
double unit_time(int whole, int half) {
    const double pairs = 1.55 * (whole / 2);
    if (whole % 2 == 0) return pairs + half_tiles_time(half);
    return pairs + (half == 0 ? 1.0 : half == 1 ? 1.2 : 2.0 + 0.45 * (half - 2));
}
double launch_time(long long whole, long long half, int ncu) {  // (in tiles)
    const int q = (int)(whole / ncu);
    const long long more = whole % ncu, fewer = ncu - more;  // compute units with q + 1 whole tiles, with q
    double t = more ? unit_time(q + 1, 0) : unit_time(q, 0);
    for (int h0 = 0, h1 = 0;;) {  // half tiles on each unit of either kind that end by t
        while (unit_time(q, h0 + 1) <= t) h0++;
        while (unit_time(q + 1, h1 + 1) <= t) h1++;
        if (h0 * fewer + h1 * more >= half) return t;
        const double t0 = unit_time(q, h0 + 1), t1 = unit_time(q + 1, h1 + 1);
        t = more && t1 < t0 ? t1 : t0;
    }
}
// Returns the time in us: 8 + 0.51 per k-group and tile (one tile or less per compute unit: 18 us at K = 1280, 26.5 at K = 2304, 107 at
// K = 12288).
double choose_row_blocks(int rows, int nblocks, int kgroups, int ncu, int *full_blocks, int *half_blocks) {
    const int units = (rows + 63) / 64, all = (units + 1) / 2;
    const long long tiles = (long long)all * nblocks;
    const int q = (int)((tiles - 1) / ncu);
    double best = launch_time(tiles, 0, ncu);
    *full_blocks = all;
    *half_blocks = 0;
    double to_beat = 0.96 * best;
    auto consider = [&](int full) {
        if (full > units / 2) full = units / 2;
        const int half = units - 2 * full;
        if (half == 0) return;
        const double t = launch_time((long long)full * nblocks, (long long)half * nblocks, ncu);
        if (t > to_beat) return;
        to_beat = t;
        best = t;
        *full_blocks = full;
        *half_blocks = half;
    };
    consider((int)((long long)q * ncu / nblocks));
    if (q >= 1) consider((int)((long long)(q - 1) * ncu / nblocks));
    if (tiles <= 2 * ncu) consider(0);
    return 8.0 + 0.51 * kgroups * best;
}

// How the tiles of an INT4 launch are laid out: split along K (kparts > 1) or in row blocks of two heights; returns the time by
// the models.
double choose_tiles_int4(const svdq_gemm_args *a, int ncu, svdq_gemm_plan *plan) {
    const int nblocks = (int)((a->N + g6::BN - 1) / g6::BN), kgroups = (int)(a->K / 64);
    double t_split;
    plan->kparts = choose_kparts((int)(a->M_pad / g6::BM) * nblocks, kgroups, ncu, &t_split);
    t_split = 0.96 * t_split + 2.8;  // (144 tiles, one per compute unit: 15.6 us at K = 1024, 33 at K = 3072, 105 at K = 12288)
    const double t_rows = choose_row_blocks(rows_needed(a), nblocks, kgroups, ncu, &plan->full_blocks, &plan->half_blocks);
    if (plan->kparts > 1 && t_split < t_rows) {
        plan->full_blocks = (int)(a->M_pad / g6::BM);
        plan->half_blocks = 0;
        return t_split;
    }
    plan->kparts = 1;
    return t_rows;
}

// Workspace: every row block's linear-attention sums; every column block's share of the next layer's low-rank projection.
size_t vk_share_bytes(const svdq_gemm_args *a, long long row_blocks) { return (size_t)row_blocks * (a->N / 96) * VK_HEAD_FLOATS * 4; }
size_t lora_share_bytes(const svdq_gemm_args *a, long long column_blocks) { return (size_t)column_blocks * a->M_pad * a->R_down * 4; }

// The argument block of the NVFP4 kernel and of the few-rows kernels.
void fill_params(const svdq_gemm_args *a, GemmParams &p) {
    p.act = (const uint8_t *)a->act;
    p.ascales = (const uint16_t *)a->ascales;
    p.wgt = (const uint8_t *)a->wgt;
    p.wscales = (const _Float16 *)a->wscales;
    p.colnorm = a->colnorm;
    p.bias = (const uint16_t *)a->bias;
    p.wcscales = (const uint16_t *)a->wcscales;
    p.lora_act = a->lora_act_in;
    p.lora_up = (const uint16_t *)a->lora_up;
    p.out = (uint16_t *)a->out;
    p.qout = (uint8_t *)a->qout;
    p.oscales = a->oscales;
    p.next_smooth_rcp = a->next_smooth_rcp;
    p.next_down = (const bf16x8_t *)a->next_lora_down;
    p.next_lora_out = a->next_lora_act_out;
    p.R_down = (int)a->R_down;
    p.M_pad = (int)a->M_pad; p.N = (int)a->N; p.K = (int)a->K;
    p.M_out = (int)a->M_out; p.N_out = (int)a->N_out; p.R_up = (int)a->R_up;
    p.alpha = a->alpha;
    for (int i = 0; i < MAX_RANK / 16; i++) p.lora_scales[i] = (a->lora_scales && i < (a->R_up + 15) / 16) ? a->lora_scales[i] : 1.0f;
    p.norm_q = (const uint16_t *)a->norm_q;
    p.norm_k = (const uint16_t *)a->norm_k;
    p.rotary = a->rotary_emb;
    p.rot_rows = (int)a->rot_rows;
    p.rope_cols = (int)(a->N / 3 * 2);
    p.norm_eps = a->norm_eps;
    p.qkv.q = (uint16_t *)a->out_q; p.qkv.k = (uint16_t *)a->out_k; p.qkv.v = (uint16_t *)a->out_v;
    p.qkv.stride_q = a->qkv_head_stride[0]; p.qkv.stride_k = a->qkv_head_stride[1]; p.qkv.stride_v = a->qkv_head_stride[2];
    p.qkv.attn_tokens = (int)a->attn_tokens; p.qkv.rows = (int)a->qkv_rows;
    p.silu = a->fuse_silu != 0;
    p.gelu = a->qout != nullptr;
    p.vk = a->out_vk;
    p.vk_rows = (int)a->vk_rows;
    p.vk_part = nullptr;
    p.next_lora_part = nullptr;
    p.partials = nullptr;
    p.counters = nullptr;
    p.whole_band = 0;
    p.row_blocks = p.full_blocks = 0;
    p.lr_steps = 0;
}

// ---- INT4: fp6 matrix instruction on the bare codes (gemm6_kernel.h) --------------------------------
void plan_int4(const svdq_gemm_args *a, int ncu, svdq_gemm_plan *plan) {
    const int kgroups = (int)(a->K / 64), all = (int)(a->M_pad / g6::BM);
    plan->full_blocks = all;
    plan->half_blocks = 0;
    plan->kparts = 1;
    if (a->k_split > 0) {
        plan->kparts = (int)(a->k_split < kgroups ? a->k_split : kgroups);
        return;
    }
    choose_tiles_int4(a, ncu, plan);
    if (a->out_vk && vk_share_bytes(a, plan->full_blocks + plan->half_blocks) > NOALLOC_SCRATCH_BYTES && vk_share_bytes(a, all) <= NOALLOC_SCRATCH_BYTES) {
        // (more row blocks, more shares: not where only 128-row blocks' fit the fixed scratch, and not in the other entry
        // point either, which gives the same bits)
        plan->full_blocks = all;
        plan->half_blocks = 0;
    }
}

void lay_out_tiles(const svdq_gemm_plan &plan, g6::Params &p) {
    p.full_blocks = plan.full_blocks;
    p.half_blocks = plan.half_blocks;
    p.kparts = plan.kparts;
    p.band = g6::band_height(p.full_blocks, 10);  // (see g6::tile_of)
    p.half_band = g6::band_height(p.half_blocks, 20);
}

int gemm_int4(const svdq_gemm_args *a, const svdq_gemm_plan &plan, hipStream_t st, int dev, bool noalloc) {
    g6::Params p;
    p.act = (const uint8_t *)a->act;
    p.ascales = (const uint16_t *)a->ascales;
    p.wgt = (const uint8_t *)a->wgt;
    p.wscales = (const uint8_t *)a->wscales;
    p.bias = (const uint16_t *)a->bias;
    p.wcscales = (const uint16_t *)a->wcscales;
    p.lora_act = a->lora_act_in;
    p.lora_up = (const uint16_t *)a->lora_up;
    p.out = (uint16_t *)a->out;
    p.qout = (uint8_t *)a->qout;
    p.oscales = (uint16_t *)a->oscales;
    p.next_smooth_rcp = a->next_smooth_rcp;
    p.next_down = (const bf16x8_t *)a->next_lora_down;
    p.next_lora_out = a->next_lora_act_out;
    p.next_lora_part = nullptr;
    p.partials = nullptr;
    p.counters = nullptr;
    p.M_pad = (int)a->M_pad; p.N = (int)a->N; p.K = (int)a->K;
    p.M_out = (int)a->M_out; p.N_out = (int)a->N_out; p.R_up = (int)a->R_up; p.R_down = (int)a->R_down;
    p.alpha = a->alpha;
    for (int i = 0; i < MAX_RANK / 16; i++) p.lora_scales[i] = (a->lora_scales && i < (a->R_up + 15) / 16) ? a->lora_scales[i] : 1.0f;
    p.norm_q = (const uint16_t *)a->norm_q;
    p.norm_k = (const uint16_t *)a->norm_k;
    p.rotary = a->rotary_emb;
    p.rot_rows = (int)a->rot_rows;
    p.rope_cols = (int)(a->N / 3 * 2);
    p.norm_eps = a->norm_eps;
    p.qkv.q = (uint16_t *)a->out_q; p.qkv.k = (uint16_t *)a->out_k; p.qkv.v = (uint16_t *)a->out_v;
    p.qkv.stride_q = a->qkv_head_stride[0]; p.qkv.stride_k = a->qkv_head_stride[1]; p.qkv.stride_v = a->qkv_head_stride[2];
    p.qkv.attn_tokens = (int)a->attn_tokens; p.qkv.rows = (int)a->qkv_rows;
    p.vk = a->out_vk;
    p.vk_rows = (int)a->vk_rows;
    p.silu = a->fuse_silu != 0;
    p.gelu = a->qout != nullptr;  // the GELU is composed exactly when the next layer's input is produced (launch_impl.cuh:282-309)

    // One workgroup per output tile (or per part of one split along K), two resident per compute unit.
    const int nblocks = (p.N + g6::BN - 1) / g6::BN;
    lay_out_tiles(plan, p);
    auto launch = [&](int nwg) { return needs_next_epilogue(a) ? g6::launch_next(p, nwg, st) : g6::launch_plain(p, nwg, st); };
    const int kparts = p.kparts, ntiles = (p.full_blocks + p.half_blocks) * nblocks;
    const size_t cnt_bytes = (size_t)ntiles * 4;
    const size_t part_bytes = kparts > 1 ? (size_t)ntiles * kparts * g6::BM * g6::BN * 4 : 0;
    const size_t share_bytes = p.next_down ? lora_share_bytes(a, nblocks) : 0;  // every column block's share of the next projection
    const size_t vk_bytes = p.vk ? vk_share_bytes(a, p.full_blocks + p.half_blocks) : 0;  // every row block's linear-attention sums
    if (kparts == 1 && !p.next_down && !p.vk) return launch(ntiles);
    std::lock_guard<std::mutex> lock(workspace_mutex(noalloc));
    const size_t cnt_pad = kparts > 1 ? (cnt_bytes + 255) & ~(size_t)255 : 0;
    WorkspaceView w;
    const size_t scratch_bytes = part_bytes + share_bytes + vk_bytes;
    if (!acquire_workspace(noalloc, dev, st, cnt_pad, scratch_bytes, &w)) return noalloc && (cnt_pad > NOALLOC_ZERO_BYTES || scratch_bytes > NOALLOC_SCRATCH_BYTES) ? SVDQ_EUNSUPPORTED : SVDQ_ELAUNCH;
    p.counters = (int *)w.zero;
    p.partials = (float *)w.scratch;
    p.next_lora_part = (float *)(w.scratch + part_bytes);
    p.vk_part = (float *)(w.scratch + part_bytes + share_bytes);
    int rc = launch(ntiles * kparts);
    if (rc == SVDQ_OK) rc = add_shares(p, rows_needed(a), nblocks, g6::BM, p.full_blocks * g6::BM, st);
    if (rc != SVDQ_OK && w.owner) w.owner->dirty = true;
    return rc;
}

// ---- NVFP4: fp16 matrix instruction on dequantized operands (gemm_kernel.h) -------------------------
// The number of workgroups that share the tiles of an NVFP4 launch out whole, where it is at least 84 % of the compute units; 0
// otherwise.
int whole_tiles_fp4(long long ntiles, int ncu) {
    long long divisor = ntiles < ncu ? ntiles : ncu;
    while (ntiles % divisor != 0) divisor--;
    return ntiles >= ncu && divisor * 100 >= ncu * 84 ? (int)divisor : 0;
}

// Persistent workgroups: one per compute unit, each walking over its share of the output tiles.
void plan_fp4(const svdq_gemm_args *a, int ncu, svdq_gemm_plan *plan) {
    const int ntiles = (int)(a->M_pad / BM) * (int)((a->N + BN - 1) / BN);
    int nwg = ntiles < ncu ? ntiles : ncu;
    int divisor = nwg;  // the largest workgroup count that divides the tile count
    while (ntiles % divisor != 0) divisor--;
    if (a->k_split == 1 || (a->k_split == 0 && whole_tiles_fp4(ntiles, ncu) > 0)) {
        // Whole tiles only: asked for, or at least 84 % of the compute units get a whole number of tiles (M = 4608,
        // N = 9216: 216 workgroups x 3 tiles 257 us, 256 even shares 256).  Then the
        // workgroups that share a block of weight columns walk K in step and find it in their L2, and no sums
        // travel through the workspace (M = 4608, N = 21504: 252 workgroups x 6 tiles 549 us, 256 even shares 560).
        nwg = divisor;
    } else if (ntiles < ncu) {
        // Fewer tiles than compute units.  A workgroup alone on its compute unit takes 1.3 us per k-group plus 12 us; the
        // parties of a tile meet through the workspace, which costs about 6 us + 13.5 us per party (measured, 12 tiles:
        // K = 3072 whole 74.6 us, two / three / four parties 63.0 / 64.0 / 69.8; K = 12288 whole 256.8, two / three /
        // four / six / eight parties 158.1 / 130.2 / 122.4 / 126.2 / 139.0).  So: whole tiles unless a split into equal
        // parts pays by that count, or the caller asks for k_split parts.  (Unasked only calls with so few tiles get here that the few-rows
        // kernel does not take: a bias, scale or factor table off its alignment.)
        const int kg = (int)(a->K / 64);
        int parties = 1;
        if (a->k_split > 1) {
            parties = (int)a->k_split;
        } else {
            double best = 1.3 * kg + 12.0;
            for (int cand : {2, 3, 4, 6, 8}) {
                if (ntiles * cand > ncu || kg / cand < 12) break;
                const double t = 1.3 * kg / cand + 6.0 + 13.5 * cand;
                if (t < (parties == 1 ? 0.90 : 0.95) * best) {  // a split has to pay clearly; more parts likewise
                    best = t;
                    parties = cand;
                }
            }
        }
        const long long units = (long long)ntiles * (a->K / 128);
        long long w = (long long)ntiles * parties;
        if (w > units) w = units;
        if (w > ncu) w = ncu;
        if (w > nwg) nwg = (int)w;
    }
    plan->workgroups = nwg;
    plan->shared_tiles = !(nwg <= ntiles && ntiles % nwg == 0);
}

int gemm_fp4(const svdq_gemm_args *a, const svdq_gemm_plan &plan, hipStream_t st, int dev, bool noalloc) {
    GemmParams p;
    fill_params(a, p);
    const int ntiles = (int)(a->M_pad / BM) * (int)((a->N + BN - 1) / BN), nwg = plan.workgroups;
    // the work is split evenly in units of two k-groups; unless the tile count is a multiple of the
    // workgroup count, some tiles are then shared by two or more workgroups and need the workspace
    const bool next = needs_next_epilogue(a);
    const bool shared_tiles = plan.shared_tiles;
    p.whole_band = 0;
    if (!shared_tiles) {
        // bands about as high as the window of an XCD's workgroups (an eighth of them) is wide, all of the same height
        // where the count allows it
        const int mblocks = p.M_pad / BM;
        int h = 1;
        while (h * h * 8 < nwg) h++;
        const int nbands = (mblocks + h - 1) / h;
        p.whole_band = (mblocks + nbands - 1) / nbands;
    }
    // every 128-column chunk's share of the next layer's low-rank projection, every row block's linear-attention sums
    const size_t share_bytes = p.next_down ? lora_share_bytes(a, a->N / 128) : 0;
    const size_t vk_bytes = p.vk ? vk_share_bytes(a, a->M_pad / 32) : 0;  // (this kernel: per 32-row slab)
    if (!shared_tiles && !share_bytes && !vk_bytes) return next ? launch_gemm_fp4_v5(p, nwg, st) : launch_gemm_fp4_v4(p, nwg, st);
    std::lock_guard<std::mutex> lock(workspace_mutex(noalloc));
    const size_t zero_bytes = shared_tiles ? (size_t)ntiles * 4 : 0, part_bytes = shared_tiles ? (size_t)2 * nwg * 256 * 64 * 16 : 0;
    const size_t scratch_bytes = part_bytes + share_bytes + vk_bytes;
    WorkspaceView w;
    if (!acquire_workspace(noalloc, dev, st, zero_bytes, scratch_bytes, &w)) return noalloc && (zero_bytes > NOALLOC_ZERO_BYTES || scratch_bytes > NOALLOC_SCRATCH_BYTES) ? SVDQ_EUNSUPPORTED : SVDQ_ELAUNCH;
    if (shared_tiles) {
        p.counters = (int *)w.zero;
        p.partials = (float *)w.scratch;
    }
    p.next_lora_part = (float *)(w.scratch + part_bytes);
    p.vk_part = (float *)(w.scratch + part_bytes + share_bytes);
    int rc = next ? launch_gemm_fp4_v5(p, nwg, st) : launch_gemm_fp4_v4(p, nwg, st);
    if (rc == SVDQ_OK) rc = add_shares(p, rows_needed(a), p.N / 128, 32, p.M_pad, st);
    if (rc != SVDQ_OK && w.owner) w.owner->dirty = true;
    return rc;
}

// ---- few rows, either precision: small tiles, operands straight to registers (gemm_direct_kernel.h) ------
struct FewRowsTile {
    int mt, nc;  // blocks of 32 rows, of 32 columns (none: large tiles)
    bool shared_rows;
    double time;
    int full_blocks;  // NVFP4, 64 x 128: blocks of 64 rows (few_rows_heights)
};
// NVFP4 launches of 64 x 128 tiles: how many blocks of 64 rows, what they leave of the rows in blocks of 32 behind them (nothing, where the last block is
// partly padding), and the time of the busiest compute unit in tiles of 64 rows.  With tiles of one height the last ones keep a few compute units busy for
// the time of a whole tile, also where most of its rows are padding; the hardware hands tiles to the emptiest compute unit, and two of them on one share
// its matrix core, so that its time is the sum of theirs.  A tile of 32 rows takes 0.68 of one of 64 (0.66 at long rows, 0.7 at K = 1024: the columns'
// operands are converted for half as many products).  Considered are whole blocks only, the last 32 rows by themselves, and 64-row tiles up to the last and
// the last but one multiple of the compute units; 1.5 % have to be gained, equal ones go to the fewest 64-row tiles.  The GEMM alone, one height / two, us, rank 32, K = 3072: norm and
// rotary, N = 9216, M = 300 21.0 / 19.2, M = 505 33.1 / 29.9, M = 700 43.5 / 40.1, M = 1200 66.3 / 63.8; quantizing, N = 12288, M = 400 40.2 / 37.0, M = 1157 97.2 / 91.9; plain, N = 3072,
// M = 2300 41.0 / 39.4.  4.5 % faster over 4600 launches of 16 ... 9216 rows (with the epilogue's requests ahead of the main loop, which came before), 6 of them slower by more than 3 %.  (Slower:
// 32-row tiles where the model sees no gain, up to 9 % where all rows are in them.  Not built for INT4, whose launches of several tiles per compute unit share the rows or are large tiles.)
// Not where tiles of 32 rows alone would be two per compute unit at most: so few are not handed to the emptiest one, and what bounds them is the requests, not the matrix core
// that the model is about.  1508 such launches are 14 % faster in 32-row tiles than in two heights, none of them slower by 4 %: SiLU, M = 67, K = 2944, N = 19840 15.7 / 18.6 us,
// quantizing, M = 65, K = 6272, N = 18176, rank 64 34.9 / 40.9.  (At three 185 launches 34 % faster.)
struct Heights {
    int full;
    double time;
};
Heights few_rows_heights(int rows, int column_blocks, int ncu) {
    constexpr double HALF = 0.68;
    const int units = (rows + 31) / 32, all = (units + 1) / 2;
    auto time = [&](int full) {
        const long long whole = (long long)full * column_blocks, half = (long long)(units - 2 * full) * column_blocks;
        const long long q = whole / ncu, more = whole % ncu, fewer = ncu - more;  // compute units with q + 1 whole tiles, with q
        for (int h0 = 0, h1 = 0;;) {  // half tiles on each unit of either kind
            const double t0 = (double)q + HALF * h0, t1 = (double)(q + 1) + HALF * h1, t = more && t1 > t0 ? t1 : t0;
            if (h0 * fewer + h1 * more >= half) return t;
            if (!more || t0 + HALF <= t1 + HALF) h0++;
            else h1++;
        }
    };
    Heights best{all, (double)(((long long)all * column_blocks + ncu - 1) / ncu)};
    if ((long long)units * column_blocks <= 2ll * ncu) return best;
    const double limit = 0.985 * best.time;
    const int q = (int)((long long)(units / 2) * column_blocks / ncu);
    for (int full : {units / 2, (int)((long long)q * ncu / column_blocks), (int)((long long)(q - 1) * ncu / column_blocks)}) {
        if (full <= 0 || full > units / 2 || 2 * full == units) continue;  // (32-row tiles alone are shape 1)
        // (the busiest compute unit has no less than all have on average)
        if (((double)full + HALF * (units - 2 * full)) * column_blocks > limit * ncu * (1.0 + 1e-9)) continue;
        const double t = time(full);
        if (t <= limit && t <= best.time) best = Heights{full, t};
    }
    return best;
}

// The tile of a few-rows launch with the plain epilogue, in blocks of 32 x 32 (`shape`: the better one of 128 columns by the models of
// choose_direct, of 32 rows (1) or 64 (2)).  What takes the time is the fetching of the operands: a
// compute unit gets 120 GB/s in requests of 16 bytes a lane, 80 in those of 8, however few of them fetch and however many waves do (48
// or 192 workgroups, 4 ... 16 waves each), and a tile of mt x nc blocks fetches mt + nc fragments per k-group.  Square tiles fetch least per
// product, small ones bring more compute units to bear: the sums cost a tile nothing before the end.  A model of the time in us, linear in the
// tiles of the busiest compute unit and in the k-groups, fitted to 844 shapes (M = 16 ... 1000, K = 1024 ... 13824, N = 1024 ... 21504)
// times the six tiles: its choice is 0.1 % (INT4) and 0.05 % (NVFP4) off the fastest on average and 5.4 % at most; tiles of 128 columns only,
// 18 and 21 %.  Measured, layer calls, 128 columns / the choice, us:
//   INT4   M = 64, K = N = 3072  13.3 / 10.2 (32 x 32)    NVFP4  14.6 / 10.3
//          M = 256               14.1 / 13.1 (64 x 64)           15.3 / 14.1
//          M = 64, K = 12288     32.3 / 21.4 (32 x 32)           34.6 / 21.6
//          M = 256, K = 12288    34.7 / 30.3 (64 x 64)           37.4 / 34.0
// Few columns, and INT4 with short rows (fewer than 1024), where 64-row tiles are the better ones of 128 columns: compute units have several tiles, and the
// model, which does not know the fixed part of a tile well, favours narrow ones too much.  There they are taken if it says 8 %, and in INT4 not
// with K = 128: M = 125, K = 128, N = 11392, rank 16 5.1 us with 64 x 128, 32 x 32 6.3; NVFP4 M = 5041, K = 8448, N = 512 48.2, 64 x 64 55.8.  Over 325 INT4 and 357 NVFP4
// shapes with few columns, short rows or more than 9216 rows 0.9 and 0.6 % off the fastest tile, without this 1.1 and 0.6; 1111 and 1370 others 0.2 and 0.3 % (M = 1 ...
// 20000, K = 128 ... 16640, N = 128 ... 21504, ranks 0 ... 160).  NVFP4, 64 x 128 tiles with 32-row ones behind them at their time: 0.3 % off over 1100 shapes, 0.7 at
// that of 64-row ones alone (M = 800, K = N = 3072 17.9 us in 64 x 64, 16.7 so).
FewRowsTile plain_tile(const svdq_gemm_args *a, int ncu, int shape, const Heights &tall) {
    struct Model {
        int mt, nc;
        double launch, tile, kgroup;
    };
    constexpr Model int4[] = {{1, 1, -0.18, 0.18, 0.0382}, {1, 2, -0.46, 0.68, 0.0551}, {2, 1, -0.46, 0.75, 0.0499},
                              {2, 2, 0.18, 0.64, 0.0702},  {1, 4, -0.13, 0.64, 0.0948}, {2, 4, 1.04, 0.53, 0.1378}};
    constexpr Model nvfp4[] = {{1, 1, -0.85, 0.16, 0.0323}, {1, 2, -0.52, 0.14, 0.0515}, {2, 1, -0.64, 0.24, 0.0498},
                               {2, 2, -0.17, 0.46, 0.0719}, {1, 4, 0.22, 0.47, 0.0876},  {2, 4, 1.96, -0.07, 0.1112}};
    const long long row_blocks = (rows_needed(a) + 31) / 32, column_blocks = a->N / 32;
    const bool favour_wide = shape == 2 && (a->N < 1024 || (!a->fp4 && a->K < 1024));
    FewRowsTile best{};
    for (const Model &m : a->fp4 ? nvfp4 : int4) {
        const bool wide = m.mt == 2 && m.nc == 4;
        if (favour_wide && !a->fp4 && a->K < 256 && !wide) continue;
        const long long tiles = (row_blocks + m.mt - 1) / m.mt * (column_blocks / m.nc);
        double rounds = (double)((tiles + ncu - 1) / ncu), launch = m.launch;
        if (a->fp4 && wide) {
            if (tall.time < rounds) launch += 0.25;  // (two heights)
            rounds = tall.time;
        }
        const double t = (launch + rounds * (m.tile + m.kgroup * (double)(a->K / 64))) * (favour_wide && wide ? 0.92 : 1.0);
        if (best.mt == 0 || t < best.time) best = FewRowsTile{m.mt, m.nc, false, t, a->fp4 && wide ? tall.full : 0};
    }
    return best;
}

// INT4 launches with more than one tile of 64 x 128 per compute unit and up to two (plain epilogue: from one and a half on): such tiles, where they are
// chosen (choose_direct), have waves that split the columns and share the rows' operands through LDS (gemm_direct_kernel.h).  A tile alone on its
// compute unit is a chain of latencies, 0.2 us per k-group, two overlap; more issue more instructions per product than the large tiles.  The GEMM alone,
// waves that split K / large tiles / this one, us, rank 32: norm and rotary M = 256, K = 3072, N = 9216 23.6 / 22.5 / 19.6, M = 505, K = 2048, N = 6144 18.0 / 17.1 / 15.7, at
// 2.25 tiles M = 505, K = 3072, N = 9216 34.6 / 29.6 / 30.6; quantizing epilogue K = 3072, N = 12288 M = 256 29.8 / 29.2 / 26.7, M = 300 30.8 / 30.4 / 28.8, at three tiles M = 505
// 43.6 / 39.4 / 39.3, rank 128 59.4 / 47.3 / 52.6; layer calls, plain M = 384, K = 3072, N = 9216 26.3 / 22.8 with this one, M = 320 (1.4 tiles, where narrow ones are better)
// 22.4 / 22.6, M = 505 30.4 / 32.1.
// Also with two and a half to (less than) three tiles per compute unit, ranks up to 64 and 1024 columns: whole large tiles are then one and a half per compute unit at best, where the
// second one doubles the time of the first.  2075 launches (K = 256 ... 16640, all epilogues) 5 % faster than large tiles, 12 % with K below 1024, 5 with N = 6144 and more at K = 8192 ... 16640 (norm and
// rotary, M = 640, K = 3072, N = 9216 27.7 / 26.4 us), 33 of them 3 to 10 % slower (half of them of 4500 to 6200 columns, 323 ... 360 large tiles).  Not with less than 2048 columns that large tiles have whole blocks of
// 256 of, and K = 1536 or more: 1.3 % slower over 197 launches, 25 of them 3 to 8 % (plain, M = 4184, K = 5376, N = 1280 42.0 / 45.3; where half of the last block is none, as at N = 1152 and 1408, 1 % faster).  Less than 1024 columns up to 14 % slower
// (linear attention, M = 15360, K = 256, N = 384 16.0 / 18.6); rank 128, whose operands do not all fit beside the stages of three
// workgroups, 8.8 % slower, above three tiles 12 to 25 % slower.  (Between two and two and a half large tiles are kept though 4 % slower: a gain that has not been
// taken yet.)
enum class SharedRows { NO, IF_FASTEST, YES };
// (`split`: the large tiles would be split along K, see choose_direct)
SharedRows staged_rows(const svdq_gemm_args *a, int ncu, bool split) {
    if (a->fp4 || a->K < 256) return SharedRows::NO;
    const long long tiles = (rows_needed(a) + 63) / 64 * (a->N / 128);
    const bool whole_blocks = a->N % 256 == 0 && a->N < 2048 && a->K >= 1536;
    if (!split && a->R_up <= 64 && a->N >= 1024 && !whole_blocks && 2 * tiles >= 5 * ncu && tiles < 3 * ncu) return SharedRows::YES;
    const bool may = 2 * tiles >= (needs_next_epilogue(a) ? 2 * ncu + 2 : 3 * ncu) && tiles <= (a->qout && split ? 3 : 2) * ncu;
    return may ? SharedRows::IF_FASTEST : SharedRows::NO;
}

// NVFP4 launches of tiles of 128 columns whose low-rank operands come through LDS (gemm_direct_kernel.h, RANKS).  They are copied 32 ranks at a time, and 16 that are left over take
// as long as 32, so an odd number of them pays only where the copies of one tile pass beside another one: wave by wave / through LDS over 15000 launches, tiles of 32 rows 0.97 at ranks 48,
// 80, 112 and 144 (silu, M = 66, K = 640, N = 2688, rank 48 6.3 / 6.7 us), 0.96 at 176 to 240, at 64 1.00, at 96 1.01, at 128 to 512 1.03 to 1.05; of 64 rows, one per compute unit 0.98 at
// 48, 0.99 at 80 and 112, 0.96 at 144 and more, several 1.00 at 48, 1.02 at 80, 1.04 at 112, 1.01 to 1.02 at 144 and more, at 64 1.02 and 1.06, at 96 1.06 and 1.12, at 128 1.09 and 1.2.
bool copies_ranks(const svdq_gemm_args *a, int ncu, int mt) {
    if (a->R_up <= 32) return false;
    return a->R_up % 32 == 0 || (a->R_up > 48 && mt == 2 && (rows_needed(a) + 63) / 64 * (a->N / 128) > ncu);
}

// Which tiles of the few-rows kernel a launch takes, if any.  Shape 1: tiles of 32 rows x 128 columns, four waves split
// K.  Shape 2: tiles of 64 rows x 128 columns, a quarter fewer operand bytes per product, from about 400 tiles of 32 rows on; INT4: two waves
// split K and two the columns, NVFP4: four waves split K.  Models of the time in us fitted to launches at K = 1024 ... 12288
// on 256 compute units, linear in the number of tiles that the busiest compute unit works through and in the k-groups; they met
// the measurements within about 10 % when they were fitted, over 2200 random shapes; what has changed since is in the terms below (NVFP4 beside whole large tiles: other models).  Measured at K = 3072 at the time of the fit, large tiles (split along K where that pays) / shape 1 / shape 2:
//   INT4   M = 256, N = 3072   22.8 /  9.6 / 12.3     NVFP4  60.7 / 11.8 / 13.8
//          M = 505, N = 9216   28.7 / 33.1 / 30.6            62.9 / 38.4 / 34.1
//          M = 1157, N = 3072  29.7 / 27.6 / 21.8            62.1 / 31.7 / 25.7
//          M = 1024, N = 9216  36.1 / 57.7 / 48.5            68.4 / 69.7 / 57.9
//          M = 1157, N = 12288                               80.1 / 103.8 / 88.6, with the quantizing epilogue 106.7 / 126.2 / 105.4
//          M = 4608, N = 12288                               298 / 407 / 317, with the quantizing epilogue 387 / 457 / 358
//   K = 12288, N = 3072: M = 256  42.1 / 24.8 / 34.4           113.6 / 30.8 / 35.0
//          M = 505             45.4 / 44.1 / 34.6           115.2 / 50.8 / 37.9
//          M = 1157            66.6 / 86.6 / 65.6           127.5 / 99.5 / 81.2
// (Since then: INT4 large tiles 3 to 10 % faster, M = 505, N = 9216 24.9, M = 1024, N = 9216 32.3; NVFP4 large tiles with the quantizing epilogue M = 1157,
// N = 12288 100; NVFP4 in the few-rows kernel M = 1157, K = 12288 76.4.)
FewRowsTile choose_direct(const svdq_gemm_args *a, int ncu) {
    constexpr FewRowsTile none{};
    if (a->k_split > 0) return none;  // (the caller asks for the tiles that k_split is about)
    if (((uintptr_t)a->bias | (uintptr_t)a->wcscales | (uintptr_t)a->oscales) % 8 || (uintptr_t)a->colnorm % 16) return none;  // (read four columns at a time)
    const bool plain = !needs_next_epilogue(a);
    const int rows = rows_needed(a), kg = (int)(a->K / 64);
    const long long ncols = a->N / 128;
    const double c1 = (double)((((rows + 31) / 32) * ncols + ncu - 1) / ncu), c2 = (double)((((rows + 63) / 64) * ncols + ncu - 1) / ncu);
    double t_large, t1, t2;
    Heights tall{};  // (worked out once a call: 20 to 70 ns of it)
    if (a->fp4) {
        const long long ntiles = (a->M_pad / BM) * ((a->N + BN - 1) / BN);
        const double tiles = (double)ntiles / ncu;
        const int nwg = whole_tiles_fp4(ntiles, ncu);
        const double own1 = a->qout ? 1.1 : a->rotary_emb ? 0.9 : 0.0, own2 = a->qout ? 1.4 : a->rotary_emb ? 1.0 : 0.0;  // of the epilogue
        auto shape2_time = [&](double tiles) { return 5.0 + tiles * (1.6 + 0.205 * kg + own2) - (tiles < 3.0 ? 0.04 * kg : 0.0); };
        // (32-row tiles behind the 64-row ones at their time: 0.2 % off the better shape over 3500 launches, 2 of them more than 10 %; at that of 64-row ones alone
        // 0.35 %, 58)
        tall = few_rows_heights(rows, (int)ncols, ncu);
        t1 = 4.3 + c1 * (1.1 + 0.127 * kg + own1);
        t2 = shape2_time(tall.time);
        if (tiles > 1.0 && !nwg) {
            // Large tiles shared by workgroups: 26 to 40 us for the sums that meet in the workspace.  (They need 128 MB of it, more than the fixed scratch
            // has, and a call gives the same bits with either: they stay where these models put them, though up to 17 % faster beyond, M = 6400, K = 640,
            // N = 16384 210 us against 181; with 64-row tiles alone beside them, as when the models were fitted.)
            t_large = (1.3 * kg + 14.0 + (a->qout ? 20.0 : a->rotary_emb ? 10.0 : 0.0)) * tiles + 33.0;
            if (t1 >= t_large && shape2_time(c2) >= t_large) return none;
            t_large = HUGE_VAL;
        } else {
            // Whole large tiles, in one round or several.  Their time and that of the few-rows kernel beside them, fitted to 555 and 400 launches in which the two are
            // within 1.6 of each other (M up to 20000, K = 128 ... 16640, ranks 0 ... 160, all epilogues): a tile's rank and epilogue cost either kernel, small
            // tiles more of it.  0.1 and 0.4 % off the faster one, 10 and 22 of them 3 % and more slower; with the models above and a factor between the kernels 1.3 and
            // 4.1 %, 70 and 130.  The GEMM alone, large tiles / few rows, us: M = 1836, K = 12032, N = 5888 256 / 199, SiLU M = 1098, K = 1792, N = 12288,
            // rank 48 63.7 / 52.2, M = 901, K = 4736, N = 11264, rank 128 115.5 / 100.5; M = 2972, K = 1792, N = 4864, rank 128 59.7 / 72.1, M = 8470, K = 1280,
            // N = 3584, rank 128 92 / 131, M = 4608, K = 3072, N = 21504 497 / 536.  Long rows: no tiling gets past the power limit, where large tiles are as fast (M = 4608,
            // K = 15360, N = 3072 322 / 325; 1.25 to 1.39 PFLOP/s in the fastest tenth of either).
            struct Model {
                double launch, tile, kgroup, rank, next, vk, rotary, silu;
                double time(const svdq_gemm_args *a, double rounds) const {
                    const double epilogue = a->qout ? next : a->out_vk ? vk : a->rotary_emb ? rotary : a->fuse_silu ? silu : 0.0;
                    return launch + rounds * (tile + kgroup * (double)(a->K / 64) + rank * (double)(a->R_up / 16) + epilogue);
                }
            };
            constexpr Model shape1{3.7, 1.06, 0.1132, 0.248, 1.37, 0.79, 0.49, 0.16};
            // Ranks above 32, whose operands come through LDS in the few-rows kernel, cost it 0.17 us per 16 ranks and tile of 64 rows, and more at K below 1536, where the copies of a tile
            // have fewer products of another to pass beside: 0.31 (large tiles in several rounds: 0.41) at K = 0.  Of 1071 launches that this brings here 31 are slower than in large tiles by 3 %
            // and more, 12 % at most; with 0.17 at any K 267 of 1500, up to 28 % (large tiles / few rows, us: plain, M = 15370, K = 128, N = 1920, rank 80 37.7 / 48.3, norm and rotary, M = 10352, K = 384, N = 3072,
            // rank 64 58.0 / 67.7).  (From rank 128 on it stands at 0.33, not fitted again.)  Ranks 0 and 16 at K = 128: by the 64-row tiles alone,
            // 32-row ones behind them gain nothing there (plain, M = 11853, K = 128, N = 1280, rank 0 14.8 / 17.4; rank 32, where large tiles take longer, N = 896, M = 12799 17.4 / 15.0).
            const double shorter = a->K < 1536 ? 1.0 - (double)a->K / 1536 : 0.0;
            auto shape2_rank = [&](double up_to_32, double short_rows) { return a->R_up <= 32 ? up_to_32 : a->R_up < 128 ? 0.17 + short_rows * shorter : 0.33; };
            const double rounds2 = a->R_up < 32 && a->K < 256 ? c2 : tall.time;
            double t_few;
            if (tiles <= 1.0) {
                const Model shape2{4.43, 1.19, 0.165, shape2_rank(0.423, 0.14), 2.48, 1.51, 0.92, 0.48};
                const Model large{6.65, 6.65, 0.344 + 1.179 * tiles, 1.23, 27.7, 15.8, 8.0, 6.4};
                t_large = large.time(a, 1.0);
                t_few = t1 < t2 ? shape1.time(a, c1) : shape2.time(a, rounds2);
            } else {
                const Model shape2{0.65, 1.394, 0.1719, shape2_rank(0.441, 0.24), 2.21, 0.99, 0.99, 0.48};
                constexpr Model large{8.14, 8.39, 1.398, 1.09, 20.0, 12.8, 8.4, 7.6};
                t_large = large.time(a, (double)(ntiles / nwg));
                t_few = t1 < t2 ? shape1.time(a, c1) : shape2.time(a, rounds2);
            }
            const double t_power = 2.0 * rows * (double)a->K * (double)a->N / 1.28e9;  // (us at 1.28 PFLOP/s)
            if (t_few < t_power) t_few = t_power;
            if (t_few >= t_large && 2 * ntiles > ncu) return none;  // (fewer would be split along K, and need workspace for their sums)
            t_large = HUGE_VAL;
        }
    } else {
        svdq_gemm_plan tiles;
        t_large = choose_tiles_int4(a, ncu, &tiles);
        t1 = 3.5 + c1 * (1.1 + 0.106 * kg);
        t2 = 3.3 + c2 * (1.6 + 0.158 * kg);
        // Tiles whose waves share the rows' operands take shape 2's place where that is the fastest by the models, and with 0.9 of its time where the others say
        // so; not against whole tiles in launches with the quantizing epilogue, whose low-rank term costs the large tiles less (rank 128, M = 1294,
        // K = 1152, N = 4608 0.85 times as fast).  Beside tiles split along K they are always taken, though those are up to 1.14 times as fast at K of
        // 8192 and more (1.06 times as slow on average): the sums need workspace, and a program may capture a call that does not without a call before.
        // Over 2500 launches of 1 ... 36864 rows with all epilogues but the plain one, ranks 0 ... 160, 0.7 % off the fastest, and 17 of them, those beside split
        // tiles, 3 % and more slower than without this form; taken wherever it can be, and with up to three tiles in MLPs, 1.0 % and 86, up to 1.4 times as slow
        // (quantizing epilogue, M = 4357, K = 1024, N = 1152, rank 128; SiLU, M = 408, K = 512, N = 4864, rank 96 8.7 us in shape 1, 12.0 so).
        const bool split = tiles.kparts > 1;
        const SharedRows shared = staged_rows(a, ncu, split);
        if (shared == SharedRows::YES) return FewRowsTile{2, 4, true};
        if (shared == SharedRows::IF_FASTEST) {
            if (split) t_large = HUGE_VAL;
            const double t = a->qout ? t2 : 0.9 * t2;
            if (t <= t1 && t < t_large) return FewRowsTile{2, 4, true};
        }
        if (plain) {
            // (the plain epilogue's tiles are faster than these two, the model of their time has no offset: 2277 layers of 100 ... 2600 rows 0.3 % off the
            // fastest, 0.6 without; M = 225, K = 4992, N = 10624 36.4 -> 30.5 us, M = 175, K = 9984, N = 14976 59 -> 51, M = 261, K = 1152, N = 14208 18 -> 17)
            const FewRowsTile t = plain_tile(a, ncu, t1 < t2 ? 1 : 2, tall);
            if (5.0 + 1.3 * t.time < t_large) return t;
            t_large *= 0.95;
        }
    }
    if ((t1 < t2 ? t1 : t2) >= t_large) return none;
    const int shape = t1 < t2 ? 1 : 2;
    return plain ? plain_tile(a, ncu, shape, tall) : FewRowsTile{shape, 4, false, 0.0, shape == 2 ? tall.full : 0};
}

// Which kernel a call takes and how it divides the work.  A function of the arguments and the number of compute units alone:
// the entry points with and without an allocation give the same bits.
void make_plan(const svdq_gemm_args *a, int ncu, svdq_gemm_plan *plan) {
    *plan = svdq_gemm_plan{};
    FewRowsTile t = choose_direct(a, ncu);
    // Its shares are those of 128 columns and 32 rows each.  Where only the shares of the INT4 kernel's larger tiles fit the fixed
    // scratch, that one is taken.  (NVFP4: the shares of both kernels are as many.)
    if (t.mt && !a->fp4) {
        auto shares = [&](int64_t column_blocks, int64_t row_blocks) {
            return (a->next_lora_down ? lora_share_bytes(a, column_blocks) : 0) + (a->out_vk ? vk_share_bytes(a, row_blocks) : 0);
        };
        if (shares(a->N / 128, a->M_pad / 32) > NOALLOC_SCRATCH_BYTES && shares((a->N + g6::BN - 1) / g6::BN, a->M_pad / g6::BM) <= NOALLOC_SCRATCH_BYTES) t = FewRowsTile{};
    }
    if (t.mt) {
        plan->few_rows = t.mt;
        plan->columns = 32 * t.nc;
        plan->shared_rows = t.shared_rows;
        plan->row_blocks = (rows_needed(a) + 32 * t.mt - 1) / (32 * t.mt);
        plan->copied_ranks = a->fp4 && t.nc == 4 && copies_ranks(a, ncu, t.mt);
        plan->full_blocks = t.full_blocks;
        const int low = (rows_needed(a) + 31) / 32 - 2 * t.full_blocks;
        plan->low_blocks = t.full_blocks && low > 0 ? low : 0;
    } else if (a->fp4) {
        plan_fp4(a, ncu, plan);
    } else {
        plan_int4(a, ncu, plan);
    }
}

int gemm_direct(const svdq_gemm_args *a, const svdq_gemm_plan &plan, hipStream_t st, int dev, bool noalloc) {
    GemmParams p;
    fill_params(a, p);
    const bool next = needs_next_epilogue(a), fp4 = a->fp4 != 0;
    const int mt = plan.few_rows;
    p.full_blocks = plan.full_blocks;
    p.row_blocks = plan.full_blocks ? plan.full_blocks + plan.low_blocks : plan.row_blocks;
    auto launch = [&]() {
        if (plan.columns < 128) return plan.columns == 32 * mt ? direct::launch_square(p, fp4, mt, st) : direct::launch_oblong(p, fp4, mt, st);
        if (plan.shared_rows) return next ? direct::launch_staged_next(p, st) : direct::launch_staged_plain(p, st);
        if (plan.copied_ranks) return next ? direct::launch_fp4_ranks_next(p, mt, st) : direct::launch_fp4_ranks_plain(p, mt, st);
        if (fp4) return next ? direct::launch_fp4_next(p, mt, st) : direct::launch_fp4_plain(p, mt, st);
        return next ? direct::launch_int4_next(p, mt, st) : direct::launch_int4_plain(p, mt, st);
    };
    // every 128-column chunk's share of the next layer's low-rank projection, every 32-row block's linear-attention sums
    const size_t share_bytes = p.next_down ? lora_share_bytes(a, a->N / 128) : 0;
    const size_t vk_bytes = p.vk ? vk_share_bytes(a, a->M_pad / 32) : 0;
    if (!share_bytes && !vk_bytes) return launch();
    std::lock_guard<std::mutex> lock(workspace_mutex(noalloc));
    WorkspaceView w;
    if (!acquire_workspace(noalloc, dev, st, 0, share_bytes + vk_bytes, &w)) return noalloc && share_bytes + vk_bytes > NOALLOC_SCRATCH_BYTES ? SVDQ_EUNSUPPORTED : SVDQ_ELAUNCH;
    p.next_lora_part = (float *)w.scratch;
    p.vk_part = (float *)(w.scratch + share_bytes);
    int rc = launch();
    if (rc == SVDQ_OK) rc = add_shares(p, rows_needed(a), p.N / 128, 32, p.M_pad, st);
    return rc;
}
}  // namespace

namespace {
int check_arguments(const svdq_gemm_args *a) {
    SVDQ_REQUIRE(a, "gemm: null args");
    SVDQ_REQUIRE(a->act && a->ascales && a->wgt && a->wscales, "gemm: act/ascales/wgt/wscales must not be null");
    SVDQ_REQUIRE(!a->fp4 || a->colnorm, "gemm: NVFP4 needs colnorm");
    SVDQ_REQUIRE(a->M_pad > 0 && a->M_pad % 256 == 0, "gemm: M_pad (%lld) must be a positive multiple of 256", (long long)a->M_pad);
    SVDQ_REQUIRE(a->N > 0 && a->N % 128 == 0, "gemm: N (%lld) must be a positive multiple of 128", (long long)a->N);
    SVDQ_REQUIRE(a->K > 0 && a->K % 128 == 0, "gemm: K (%lld) must be a positive multiple of 128", (long long)a->K);
    SVDQ_REQUIRE(a->out || a->qout || a->out_q, "gemm: one of out / qout / out_q must be given");
    SVDQ_REQUIRE((a->lora_up != nullptr) == (a->lora_act_in != nullptr), "gemm: lora_up and lora_act_in go together");
    SVDQ_REQUIRE(a->R_up >= 0 && a->R_up % 16 == 0 && a->R_up <= MAX_RANK, "gemm: R_up (%lld) must be a multiple of 16, at most %d", (long long)a->R_up, MAX_RANK);
    SVDQ_REQUIRE((a->R_up > 0) == (a->lora_up != nullptr), "gemm: R_up and lora_up disagree");
    SVDQ_REQUIRE(a->k_split >= 0, "gemm: k_split must not be negative");
    SVDQ_REQUIRE(a->M_out >= 0 && a->M_out <= a->M_pad, "gemm: M_out (%lld) does not fit M_pad (%lld)", (long long)a->M_out, (long long)a->M_pad);
    if (a->out) {
        SVDQ_REQUIRE(a->M_out > 0 && a->M_out <= a->M_pad && a->M_pad - a->M_out < 256, "gemm: M_out (%lld) does not fit M_pad (%lld)",
                     (long long)a->M_out, (long long)a->M_pad);
        if (a->out_vk) {
            SVDQ_REQUIRE(a->N_out * 3 == a->N && a->M_out == a->M_pad, "gemm: with out_vk, `out` is the q third of all rows: [M_pad, N/3]");
        } else {
            SVDQ_REQUIRE(a->N_out > 0 && a->N_out <= a->N && a->N - a->N_out < 128 && a->N_out % 8 == 0,
                         "gemm: N_out (%lld) must be a multiple of 8 within 128 of N (%lld)", (long long)a->N_out, (long long)a->N);
        }
    }
    if (a->out_vk) {
        // EpilogueLiteLA (gemm_w4a4_launch_impl.cuh:311-345)
        SVDQ_REQUIRE(a->out && !a->qout && !a->rotary_emb && !a->next_lora_down && !a->fuse_silu, "gemm: out_vk goes with `out` (the q third) alone");
        SVDQ_REQUIRE(a->N % 384 == 0, "gemm: out_vk needs N (%lld) to be three equal parts of whole 128-column blocks", (long long)a->N);
        SVDQ_REQUIRE(a->vk_rows > 0 && a->vk_rows % 256 == 0 && a->M_pad % a->vk_rows == 0,
                     "gemm: vk_rows (%lld) must be a multiple of 256 that divides M_pad (%lld)", (long long)a->vk_rows, (long long)a->M_pad);
        SVDQ_REQUIRE((uintptr_t)a->out_vk % 16 == 0, "gemm: out_vk must be 16-byte aligned");
    }
    SVDQ_REQUIRE(((uintptr_t)a->act | (uintptr_t)a->wgt | (uintptr_t)a->ascales | (uintptr_t)a->wscales | (uintptr_t)a->out |
                  (uintptr_t)a->lora_act_in | (uintptr_t)a->lora_up) % 16 == 0, "gemm: pointers must be 16-byte aligned");
    SVDQ_REQUIRE(a->M_pad * a->N < (1ll << 40) && a->K < (1 << 24), "gemm: shape too large");
    // scale tables are addressed with 32-bit lane offsets
    SVDQ_REQUIRE((a->K / 64) * a->M_pad * 4 < (1ll << 31) && (a->K / 64) * a->N * 8 < (1ll << 31), "gemm: scale tables too large");
    // SiLU goes with the plain store only (gemm_w4a4_launch_impl.cuh:404-417)
    if (a->fuse_silu && (a->qout || a->rotary_emb || !a->out)) return fail(SVDQ_EUNSUPPORTED, "gemm: fuse_silu goes with `out` alone (no qout, no rotary_emb)");
    if (a->fp4 && a->act_unsigned) return fail(SVDQ_EINVAL, "gemm: NVFP4 activations are never unsigned");
    if (a->qout) {
        SVDQ_REQUIRE(a->oscales && a->next_smooth_rcp, "gemm: qout needs oscales and next_smooth_rcp");
        SVDQ_REQUIRE(((uintptr_t)a->qout | (uintptr_t)a->next_smooth_rcp) % 16 == 0, "gemm: qout pointers must be 16-byte aligned");
    }
    SVDQ_REQUIRE((a->next_lora_down != nullptr) == (a->next_lora_act_out != nullptr) && (a->next_lora_down != nullptr) == (a->R_down > 0),
                 "gemm: next_lora_down, next_lora_act_out and R_down go together");
    SVDQ_REQUIRE(a->R_down >= 0 && a->R_down % 16 == 0 && a->R_down <= MAX_RANK, "gemm: R_down (%lld) must be a multiple of 16, at most %d", (long long)a->R_down, MAX_RANK);

    if (a->rotary_emb) {
        SVDQ_REQUIRE(a->norm_q && a->norm_k, "gemm: rotary_emb needs norm_q and norm_k");
        SVDQ_REQUIRE(a->N % 384 == 0, "gemm: rotary_emb needs N (%lld) to be three equal parts of 128-wide heads", (long long)a->N);
        SVDQ_REQUIRE(!a->qout, "gemm: rotary_emb goes without qout");
        const long long covered = a->out_q ? a->attn_tokens : a->M_out;
        if (a->out_q) {
            // EpiloguePackQKV in place of the plain store (gemm_w4a4_launch_impl.cuh:380-397)
            SVDQ_REQUIRE(!a->out && a->out_k && a->out_v, "gemm: out_q, out_k and out_v go together, without `out`");
            SVDQ_REQUIRE(a->qkv_rows > 0 && a->qkv_rows <= a->M_pad && a->attn_tokens >= 0 && a->attn_tokens <= a->qkv_rows,
                         "gemm: attn_tokens (%lld) <= qkv_rows (%lld) <= M_pad (%lld) does not hold", (long long)a->attn_tokens,
                         (long long)a->qkv_rows, (long long)a->M_pad);
            SVDQ_REQUIRE(a->qkv_head_stride[0] >= a->qkv_rows * 128 && a->qkv_head_stride[1] >= a->qkv_rows * 128 && a->qkv_head_stride[2] >= a->qkv_rows * 128,
                         "gemm: a head of out_q / out_k / out_v holds qkv_rows x 128 values, the head strides are smaller");
            SVDQ_REQUIRE(a->qkv_head_stride[0] % 8 == 0 && a->qkv_head_stride[1] % 8 == 0 && a->qkv_head_stride[2] % 8 == 0 &&
                             ((uintptr_t)a->out_q | (uintptr_t)a->out_k | (uintptr_t)a->out_v) % 16 == 0,
                         "gemm: out_q / out_k / out_v and their head strides must be 16-byte aligned");
        } else {
            SVDQ_REQUIRE(a->out && a->N_out == a->N, "gemm: rotary_emb goes with a full-width `out` (or with out_q, out_k, out_v)");
        }
        // (the kernels read the last block of the table for rows beyond it: an empty table has none)
        SVDQ_REQUIRE(a->rot_rows > 0 && a->rot_rows >= covered && a->rot_rows <= a->M_pad && a->rot_rows % 32 == 0,
                     "gemm: rotary_emb has %lld rows for %lld output rows (must cover them, in whole blocks of 32)", (long long)a->rot_rows, covered);
        SVDQ_REQUIRE(((uintptr_t)a->rotary_emb % 16 == 0) && ((uintptr_t)a->norm_q % 8 == 0) && ((uintptr_t)a->norm_k % 8 == 0),
                     "gemm: rotary_emb / norm pointers are not aligned");
    } else {
        SVDQ_REQUIRE(!a->norm_q && !a->norm_k, "gemm: norm_q / norm_k need rotary_emb");
        SVDQ_REQUIRE(!a->out_q && !a->out_k && !a->out_v, "gemm: out_q / out_k / out_v need rotary_emb (the reference composes them only there)");
    }

    return SVDQ_OK;
}

int gemm_entry(const svdq_gemm_args *a, void *stream, bool noalloc) {
    const int rc = check_arguments(a);
    if (rc != SVDQ_OK) return rc;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return fail(SVDQ_ELAUNCH, "gemm: cannot identify the current device");
    const int ncu = compute_units(dev);
    if (ncu <= 0) return fail(SVDQ_ELAUNCH, "gemm: cannot query the number of compute units");
    svdq_gemm_plan plan;
    make_plan(a, ncu, &plan);
    if (plan.few_rows) return gemm_direct(a, plan, (hipStream_t)stream, dev, noalloc);
    return a->fp4 ? gemm_fp4(a, plan, (hipStream_t)stream, dev, noalloc) : gemm_int4(a, plan, (hipStream_t)stream, dev, noalloc);
}
}  // namespace

namespace {
// `M_out` without `out` is the number of rows to work out (rows_needed): not a caller's to set, it is the shape of `out`
int public_entry(const svdq_gemm_args *a, void *stream, bool noalloc) {
    if (!a || a->out || a->M_out == 0) return gemm_entry(a, stream, noalloc);
    svdq_gemm_args all = *a;
    all.M_out = 0;
    return gemm_entry(&all, stream, noalloc);
}
}  // namespace

extern "C" int svdq_gemm_w4a4(const svdq_gemm_args *a, void *stream) { return public_entry(a, stream, false); }

extern "C" int svdq_gemm_w4a4_noalloc(const svdq_gemm_args *a, void *stream) { return public_entry(a, stream, true); }

extern "C" int svdq_gemm_w4a4_rows(const svdq_gemm_args *a, int64_t rows, int noalloc, void *stream) {
    SVDQ_REQUIRE(a && !a->out && rows > 0, "gemm: rows go with a call without `out`");
    svdq_gemm_args some = *a;
    some.M_out = rows;
    return gemm_entry(&some, stream, noalloc != 0);
}

extern "C" int svdq_gemm_plan_of(const svdq_gemm_args *a, int64_t rows, int compute_units, svdq_gemm_plan *plan) {
    SVDQ_REQUIRE(a && plan && compute_units > 0 && rows >= 0 && !(a->out && rows), "gemm: rows go with a call without `out`");
    svdq_gemm_args some = *a;
    if (!a->out) some.M_out = rows;
    const int rc = check_arguments(&some);
    if (rc == SVDQ_OK) make_plan(&some, compute_units, plan);
    return rc;
}

extern "C" void svdq_gemm_int4_tile(const svdq_gemm_plan *plan, int64_t N, int block, svdq_gemm_tile *tile) {
    const int nblocks = (int)((N + g6::BN - 1) / g6::BN);
    g6::Params p;
    lay_out_tiles(*plan, p);
    const g6::TileOf t = g6::tile_of(p, block, (p.full_blocks * p.kparts + p.half_blocks) * nblocks, nblocks);
    const int rows = t.whole ? g6::BM : g6::BM / 2, before = t.whole ? 0 : plan->full_blocks;
    *tile = svdq_gemm_tile{before * g6::BM + t.row_block * rows, rows, t.column_block, t.part, before + t.row_block, t.tile};
}

// (as gemm_direct_kernel takes them)
extern "C" int svdq_gemm_few_rows_tile(const svdq_gemm_plan *plan, int64_t N, int block, svdq_gemm_tile *tile) {
    const int column_blocks = (int)(N / plan->columns), full = plan->full_blocks * column_blocks;
    const int total = (plan->full_blocks ? plan->full_blocks + plan->low_blocks : plan->row_blocks) * column_blocks;
    const bool low = plan->full_blocks && block >= full;
    const int blocks = low ? plan->low_blocks : plan->full_blocks ? plan->full_blocks : plan->row_blocks, mt = low ? 1 : plan->few_rows;
    const int v = low ? direct::tile_of(block - full, total - full) : direct::tile_of(block, plan->full_blocks ? full : total), nb = v / blocks, mb = v - nb * blocks;
    *tile = svdq_gemm_tile{(low ? plan->full_blocks * 64 : 0) + mb * mt * 32, mt * 32, nb, 0, (low ? plan->full_blocks : 0) + mb, (low ? full : 0) + v};
    return total;
}

extern "C" int svdq_release_workspaces(void) {
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    int prev = 0;
    if (hipGetDevice(&prev) != hipSuccess) return fail(SVDQ_ELAUNCH, "release_workspaces: cannot identify the current device");
    int rc = SVDQ_OK;
    auto release = [&](int dev, void *ptr) {
        if (!ptr) return;
        // everything enqueued on the block's device has finished before the block goes
        if (hipSetDevice(dev) != hipSuccess || hipDeviceSynchronize() != hipSuccess || hipFree(ptr) != hipSuccess) {
            (void)hipGetLastError();
            rc = fail(SVDQ_ELAUNCH, "release_workspaces: cannot free a block on device %d", dev);
        }
    };
    for (Workspace &w : g_ws) release(w.dev, w.ptr);
    for (Retired &r : g_retired) release(r.dev, r.ptr);
    g_ws.clear();
    g_retired.clear();
    (void)hipSetDevice(prev);
    return rc;
}
