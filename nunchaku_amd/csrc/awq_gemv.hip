// AWQ W4A16 GEMV: out[m, n] = sum_k bf16(code[n, k] * scale[k/64, n] + zero[k/64, n]) * x[m, k] for m <= 8 rows.
// Counterpart of gemv_kernel (src/kernels/awq/gemv_awq.cu:84-215) behind ops.gemv_awq
// (nunchaku/csrc/pybind.cpp, nunchaku/ops/gemv.py), used by AWQW4A16Linear (nunchaku/models/linear.py:138-208).
//
// HBM-bound: every weight byte is read once.  The kernel reads the reference's storage as it is (no
// repack): per 4 output rows and 64 input channels a block of 128 bytes, 32 bytes per row
// (nunchaku/models/text_encoders/tinychat_utils.py:76-106).  Word i2 of a row's 16 bytes of a 32-channel half,
// nibble p + 4 b, is channel 8 p + 2 i2 + b: the nibbles p and p + 4 are a pair of neighbouring channels, which
// after dequantization is one packed bf16 pair, and the four pairs of one p are eight consecutive channels.
#include "svdq_common.h"

using namespace svdq;

namespace {

struct AwqParams {
    const uint16_t *x;       // bf16 [M, K]
    const uint8_t *qweight;  // reference storage, [N/4][K/64][4 rows][32 bytes]
    const uint16_t *scales;  // bf16 [K/64, N]
    const uint16_t *zeros;   // bf16 [K/64, N]
    const uint16_t *bias;    // bf16 [N] or null
    uint16_t *out;           // bf16 [M, N]
    int M, N, K;
};


// 32 codes of one channel, the 16 bytes a lane holds of a 32-channel half, to the second operands of four
// v_mfma_f32_16x16x32_bf16: operand q holds bf16(code * scale + zero) of input channels 8 q ... 8 q + 7.  A code as a byte is
// the E4M3 pattern of code * 2^-9 (subnormals and the first binade are evenly spaced), so the hardware conversion makes two
// floats per instruction, and its scale operand, 2^9, makes them the codes themselves: the scale is used as it is stored (512
// times it is infinite from 2^119 on) and the sum is rounded once, by the fused multiply-add, before the rounding to bf16.
// (One v_cvt_f32_ubyte per code: 11.1 us against 10.0 at K = 3072, N = 18432, one row, the kernel being bound by its vector
// instructions.)
__device__ inline void dequantize32(u32x4_t w, float scale, float zero, u32x4_t (&wb)[4]) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    float f[4][8];  // word i2, nibble p + 4 b = channel 8 p + 2 i2 + b
#pragma unroll
    for (int i2 = 0; i2 < 4; i2++) {
        const uint32_t even = w[i2] & 0x0F0F0F0Fu, odd = (w[i2] >> 4) & 0x0F0F0F0Fu;
        const f32x2_t e0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, false), e1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, true);
        const f32x2_t o0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, false), o1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, true);
        f[i2][0] = e0[0]; f[i2][2] = e0[1]; f[i2][4] = e1[0]; f[i2][6] = e1[1];
        f[i2][1] = o0[0]; f[i2][3] = o0[1]; f[i2][5] = o1[0]; f[i2][7] = o1[1];
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
        for (int i2 = 0; i2 < 4; i2++) wb[q][i2] = pack_bf16x2(__builtin_fmaf(f[i2][q], scale, zero), __builtin_fmaf(f[i2][q + 4], scale, zero));
}

// the reference stores bf16 and adds the bias to that (linear.py:183-185): two roundings
__device__ inline void store_result(const AwqParams &p, int m, int row, float sum) {
    float o = bf16_bits_to_f32(f32_to_bf16_bits(sum));
    if (p.bias) o = bf16_bits_to_f32(f32_to_bf16_bits(o + bf16_bits_to_f32(p.bias[row])));
    p.out[(size_t)m * p.N + row] = (uint16_t)f32_to_bf16_bits(o);
}

// K up to 4096: one workgroup of eight waves per compute unit, each wave with SPW steps of 128 input channels
// (wave, wave + 8, ...) whose activations stay in its registers for all the tiles of 16 output channels the workgroup
// walks through; the codes, scales and zeros of the next AHEAD tiles are requested while one is multiplied.  Lane l holds
// output channel l % 16 of the tile and input channels 32 (l / 16) + [0, 32) of a step: the second operand of four matrix
// instructions as dequantized (above), the first being x[m = l % 16] of the same channels, zero for rows beyond M and
// channels beyond K.  The result tile has channel l % 16 and rows 4 (l / 16) + [0, 4) in lane l; the waves' tiles meet in
// LDS once per BATCH tiles and are added in ascending order.
// Per step and wave this leaves about 85 vector instructions for 32 codes per lane, where a workgroup per tile, with its
// activations in LDS, needed 140.  Measured with weights from HBM (12 layers in turn), before / now: K = 3072,
// N = 18432 one row 11.9 / 10.7 us, four 13.0 / 10.8, eight 15.7 / 11.4; K = 4096, N = 20480, eight rows 24.1 / 15.3;
// K = 3072, N = 9216, one row 8.5 / 8.0.  About 3 us of that are launch and latency, the rest 4.2 TB/s.  Further ahead is slower
// (three tiles 11.7, four 12.4), two workgroups of half the tiles per compute unit too (13.0).
// Equal shares of the channels (N = 18432 is 4.5 tiles per workgroup, which were 4 or 5), no requests behind a share's end (the tiles
// requested ahead made 40 % more of them) and one division in place of two of 64 bits, in a graph of layers in turn that hold 520 MB together,
// twice the memory-side cache, before / now: K = 3072, N = 18432 one row 10.5 / 10.1 us (3.1 TB/s), four 10.7 / 10.7, eight 11.5 / 11.2; N = 9216
// 7.9 / 7.4; N = 3072, four rows 5.5 / 5.0; K = 4096, N = 20480 13.5 / 13.2, eight rows 15.0 / 14.4; K = 1024, N = 2048 3.3 / 3.1.  One layer again and again
// (its weights in that cache): K = 3072, N = 18432 8.4 / 8.2, 9.6 / 9.4 and 10.1 / 9.9.
constexpr int WAVES = 8, BATCH = 6, AHEAD = 2;
static_assert(BATCH % (AHEAD + 1) == 0, "the ring of register sets is indexed by the position in a batch");
template <int SPW>
__global__ void __launch_bounds__(64 * WAVES, 2) awq_gemv_rows_kernel(AwqParams p) {
    __shared__ float4_t red[BATCH][WAVES][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, kb = lane >> 4;
    const int kblocks = p.K / 64;
    int wg = blockIdx.x;
    if (gridDim.x % 8 == 0) wg = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;  // neighbours in N on one XCD: they share lines of scales
    // The workgroup's channels, in units of the storage's four; tile t holds 16 of them from c_begin + 16 t on, the last one what is left.
    const int share = (int)((unsigned)(p.N / 4) / gridDim.x), more = p.N / 4 - share * (int)gridDim.x;
    const int c_begin = 4 * (wg * share + (wg < more ? wg : more)), c_end = c_begin + 4 * (share + (wg < more ? 1 : 0));
    const int t_end = (c_end - c_begin + 15) / 16;

    u32x4_t x[SPW][4];
    uint32_t w_off[SPW], s_off[SPW];
    bool live[SPW];  // the lane's channels of the step exist
#pragma unroll
    for (int j = 0; j < SPW; j++) {
        const int cb = (wave + WAVES * j) * 2 + (kb >> 1), block = cb < kblocks ? cb : kblocks - 1;  // the lane's 64-channel block
        live[j] = cb < kblocks;
        const uint16_t *xp = p.x + (size_t)(n < p.M ? n : 0) * p.K + block * 64 + 32 * (kb & 1);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const u32x4_t v = *(const u32x4_t *)(xp + 8 * q);
            x[j][q] = live[j] && n < p.M ? v : u32x4_t{0, 0, 0, 0};
        }
        w_off[j] = (uint32_t)(n >> 2) * (uint32_t)(kblocks * 128) + (uint32_t)(n & 3) * 32u + (uint32_t)(kb & 1) * 16u + (uint32_t)block * 128u;
        s_off[j] = (uint32_t)block * (uint32_t)p.N * 2u + (uint32_t)n * 2u;
    }
    struct Tile {
        u32x4_t w[SPW];
        uint16_t s[SPW], z[SPW];
    };
    // Requests are branch-free: a lane whose channel lies behind the workgroup's last one (the end of its last tile, and the tiles
    // requested ahead at the end) gets an offset beyond its buffer, which reads zeros and touches no memory.
    const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(p.qweight + (size_t)(c_begin >> 2) * kblocks * 128), 0, ((c_end - c_begin) >> 2) * kblocks * 128, 0x00020000);
    const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc((void *)p.scales, 0, kblocks * p.N * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t zrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)p.zeros, 0, kblocks * p.N * 2, 0x00020000);
    auto load = [&](int t, Tile &d) {
        const uint32_t beyond = c_begin + 16 * t + n < c_end ? 0u : 0x80000000u;
        const int wt = t * kblocks * 512, st = (c_begin + 16 * t) * 2;
#pragma unroll
        for (int j = 0; j < SPW; j++) {
            d.w[j] = __builtin_amdgcn_raw_buffer_load_b128(wrsrc, w_off[j] | beyond, wt, 2);  // (2: a streaming load)
            d.s[j] = __builtin_amdgcn_raw_buffer_load_b16(srsrc, s_off[j] | beyond, st, 0);
            d.z[j] = __builtin_amdgcn_raw_buffer_load_b16(zrsrc, s_off[j] | beyond, st, 0);
        }
    };
    Tile ring[AHEAD + 1];
#pragma unroll
    for (int a = 0; a < AHEAD; a++) load(a, ring[a]);
    for (int t0 = 0; t0 < t_end; t0 += BATCH) {
        const int count = t_end - t0 < BATCH ? t_end - t0 : BATCH;
        if (t0 > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < BATCH; i++) {
            if (i >= count) continue;
            load(t0 + i + AHEAD, ring[(i + AHEAD) % (AHEAD + 1)]);
            __builtin_amdgcn_sched_barrier(0);
            const Tile &d = ring[i % (AHEAD + 1)];
            float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < SPW; j++) {
                u32x4_t wb[4];
                // (channels beyond K have weights of zero: the repeated block's may be infinite, and zero times that is no zero)
                dequantize32(d.w[j], live[j] ? bf16_bits_to_f32(d.s[j]) : 0.f, live[j] ? bf16_bits_to_f32(d.z[j]) : 0.f, wb);
#pragma unroll
                for (int q = 0; q < 4; q++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[j][q]), __builtin_bit_cast(bf16x8_t, wb[q]), acc, 0, 0, 0);
            }
            red[i][wave][lane] = acc;
        }
        __syncthreads();
        for (int idx = threadIdx.x; idx < count * 16 * p.M; idx += 64 * WAVES) {
            const int c = idx & 15, m = (idx >> 4) % p.M, i = (idx >> 4) / p.M;
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; w++) sum += ((const float *)&red[i][w][(m >> 2) * 16 + c])[m & 3];
            const int channel = c_begin + 16 * (t0 + i) + c;
            if (channel < c_end) store_result(p, m, channel, sum);
        }
    }
}

// Longer rows: a workgroup of four waves owns 16 output channels; the waves take the 128-channel steps of K in turn, with
// the activations in LDS where they fit.
template <bool XLDS>
__global__ void __launch_bounds__(256) awq_gemv_mfma_kernel(AwqParams p) {
    extern __shared__ u32x4_t xlds[];  // XLDS (x fits: up to 64 KB): [M][K] bf16; then, always, 4 waves x 64 lanes x float4
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t xquads = XLDS ? (size_t)p.M * p.K / 8 : 0;
    if (XLDS) {
        for (int i = threadIdx.x; i < (int)xquads; i += 256) xlds[i] = ((const u32x4_t *)p.x)[i];
        __syncthreads();
    }
    int wg = blockIdx.x;
    if (gridDim.x % 8 == 0) wg = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;  // neighbours in N on one XCD: they share lines of scales
    const int n = lane & 15, kb = lane >> 4;
    const int row_raw = wg * 16 + n;
    const int row = row_raw < p.N ? row_raw : p.N - 1;  // a channel beyond N repeats the last one and is not stored
    const int kblocks = p.K / 64;
    const int steps = (p.K + 127) / 128;
    const uint8_t *wrow = p.qweight + ((size_t)(row >> 2) * kblocks * 4 + (row & 3)) * 32 + (kb & 1) * 16;  // + 128 per 64-channel block
    const bool xrow = n < p.M;  // this lane supplies row n of x to the first operand

    constexpr int DEPTH = 3;
    u32x4_t wq[DEPTH + 1];
    uint16_t sq[DEPTH + 1], zq[DEPTH + 1];
    auto block_of = [&](int it) {  // the lane's 64-channel block in step it, clamped to the last valid one
        const int cb = it * 2 + (kb >> 1);
        return cb < kblocks ? cb : kblocks - 1;
    };
    auto load_w = [&](int it, int slot) {
        const int cb = block_of(it);
        wq[slot] = __builtin_nontemporal_load((const u32x4_t *)(wrow + (size_t)cb * 128));
        sq[slot] = p.scales[(size_t)cb * p.N + row];
        zq[slot] = p.zeros[(size_t)cb * p.N + row];
    };
    float4_t acc = {0.f, 0.f, 0.f, 0.f};
    auto step = [&](int it, int slot) {
        const bool ok = it * 2 + (kb >> 1) < kblocks;
        const u32x4_t w = wq[slot];
        const float s = ok ? bf16_bits_to_f32(sq[slot]) : 0.f, z = ok ? bf16_bits_to_f32(zq[slot]) : 0.f;
        load_w(it + 4 * DEPTH, slot == 0 ? DEPTH : slot - 1);
        const int k0 = block_of(it) * 64 + 32 * (kb & 1);
        u32x4_t xa[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            xa[j] = u32x4_t{0, 0, 0, 0};
            if (xrow) {
                const size_t xoff = (size_t)n * p.K + k0 + 8 * j;
                xa[j] = XLDS ? xlds[xoff / 8] : *(const u32x4_t *)(p.x + xoff);
            }
        }
        u32x4_t wb[4];
        dequantize32(w, s, z, wb);
#pragma unroll
        for (int q = 0; q < 4; q++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, xa[q]), __builtin_bit_cast(bf16x8_t, wb[q]), acc, 0, 0, 0);
    };
    // wave w takes the steps w, w + 4, ...; the ring of DEPTH + 1 register sets is indexed statically
#pragma unroll
    for (int d = 0; d < DEPTH; d++) load_w(wave + 4 * d, d);
    for (int it0 = wave; it0 < steps; it0 += 4 * (DEPTH + 1)) {
#pragma unroll
        for (int sl = 0; sl <= DEPTH; sl++) {
            if (it0 + 4 * sl >= steps) goto done;
            step(it0 + 4 * sl, sl);
        }
    }
done:
    float4_t *red = (float4_t *)(xlds + xquads);
    red[wave * 64 + lane] = acc;
    __syncthreads();
    if (wave == 0) {
        const float4_t a1 = red[64 + lane], a2 = red[128 + lane], a3 = red[192 + lane];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int m = 4 * kb + i;
            if (m < p.M && row_raw < p.N) store_result(p, m, row, ((acc[i] + a1[i]) + a2[i]) + a3[i]);
        }
    }
}

template <int SPW>
int launch_rows(const AwqParams &p, hipStream_t stream) {
    int dev = 0;
    const int ncu = hipGetDevice(&dev) == hipSuccess && compute_units(dev) > 0 ? compute_units(dev) : 256;
    const int ntiles = (p.N + 15) / 16;
    SVDQ_LAUNCH((awq_gemv_rows_kernel<SPW>), dim3(ntiles < ncu ? ntiles : ncu), dim3(64 * WAVES), 0, stream, p);
    return check_launch("awq_gemv_w4a16");
}

int launch_mfma(const AwqParams &p, hipStream_t stream) {
    const size_t xbytes = (size_t)p.M * p.K * 2, red = 4 * 64 * 16;
    const dim3 grid((p.N + 15) / 16);
    if (xbytes <= 64 * 1024) {
        auto kern = awq_gemv_mfma_kernel<true>;
        if (xbytes + red > 48 * 1024) {
            hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(xbytes + red));
            if (e != hipSuccess) return fail(SVDQ_ELAUNCH, "awq_gemv: cannot reserve %zu bytes of LDS: %s", xbytes + red, hipGetErrorString(e));
        }
        SVDQ_LAUNCH(kern, grid, dim3(256), xbytes + red, stream, p);
    } else {
        SVDQ_LAUNCH((awq_gemv_mfma_kernel<false>), grid, dim3(256), red, stream, p);
    }
    return check_launch("awq_gemv_w4a16");
}

}  // namespace

extern "C" int svdq_awq_gemv_w4a16(const svdq_awq_gemv_args *a, void *stream) {
    SVDQ_REQUIRE(a, "awq_gemv: null args");
    SVDQ_REQUIRE(a->x && a->qweight && a->scales && a->zeros && a->out, "awq_gemv: x/qweight/scales/zeros/out must not be null");
    SVDQ_REQUIRE(a->M > 0 && a->M <= 8, "awq_gemv: M (%lld) must be in 1..8", (long long)a->M);  // gemv_awq.cu:262
    SVDQ_REQUIRE(a->N > 0 && a->N % 4 == 0, "awq_gemv: N (%lld) must be a positive multiple of 4", (long long)a->N);
    SVDQ_REQUIRE(a->K > 0 && a->K % 64 == 0 && a->K < (1 << 24), "awq_gemv: K (%lld) must be a positive multiple of 64", (long long)a->K);
    SVDQ_REQUIRE(a->N < (1ll << 28), "awq_gemv: shape too large");
    if (a->group_size != 64) return fail(SVDQ_EUNSUPPORTED, "awq_gemv: group_size %d (only 64 is supported, as in the reference)", a->group_size);  // gemv_awq.cu:263
    SVDQ_REQUIRE(((uintptr_t)a->x | (uintptr_t)a->qweight) % 16 == 0, "awq_gemv: x and qweight must be 16-byte aligned");
    AwqParams p{(const uint16_t *)a->x, (const uint8_t *)a->qweight, (const uint16_t *)a->scales, (const uint16_t *)a->zeros,
                (const uint16_t *)a->bias, (uint16_t *)a->out, (int)a->M, (int)a->N, (int)a->K};
    hipStream_t st = (hipStream_t)stream;
    // Short rows (up to 4 steps of K) and more than 16384 channels: half of the eight waves have nothing to multiply, and many
    // workgroups of four waves are faster than few with several tiles one after the other (N = 21504, eight rows: K = 256 5.3 us against
    // 6.0, K = 384 5.6 against 6.0; K = 640 6.9 against 6.2, and the same on either side at N = 12288).
    // (byte offsets of a lane's scales are 32 bits wide)
    const int64_t steps = (a->K + 127) / 128;
    const bool rows = a->N >= 16 && steps <= 4 * WAVES && (steps > 4 || a->N <= 16384);
    if (rows && a->K / 64 * a->N < (1ll << 30)) {
        if (steps <= WAVES) return launch_rows<1>(p, st);
        if (steps <= 2 * WAVES) return launch_rows<2>(p, st);
        if (steps <= 3 * WAVES) return launch_rows<3>(p, st);
        return launch_rows<4>(p, st);
    }
    return launch_mfma(p, st);
}
