"""Host-side model of the global addresses that the INT4 GEMM kernel, the low-rank term of the NVFP4 GEMM kernel, the few-rows GEMM
kernel, the quantize kernel and the AWQ GEMV kernel form, checked against the sizes of the buffers the operators are given (CPU only;
nothing here touches a GPU).

Which tile a workgroup takes is asked of the library (``plan_util``).  The model restates the index arithmetic of
``csrc/gemm6_kernel.h`` (k-parts, the schedule of the asynchronous copies with its look-ahead, the copies of the low-rank operands,
parked partial sums, output stores), of ``csrc/gemm_kernel.h`` (low-rank operands), of ``csrc/gemm_direct_kernel.h`` (operands of both
precisions, NVFP4 ones as buffers), of ``csrc/quantize.hip`` (the row buffer whose size ends at the last valid row, code / scale /
projection stores) and of ``csrc/awq_gemv.hip`` (the shares' buffers) for whole grids, over the shape distribution of
``tests/test_gpu_shape_sweep.py`` and of the randomized loop that once ended in a GPU fault (M = 100, K = 3072, N = 768,
rank 0, three k-parts among them).  It guards the arithmetic; the fault itself came from the compiler keeping a carry flag
alive across an inline-asm statement that overwrote it (``tests/test_build_guard.py`` checks the generated code for that).

Buffer requests (a descriptor, a lane's offset and a scalar offset) are modelled with a range check that counts the scalar offset and
with one that does not: what a lane reads must not depend on it, and no sum may pass 4 GB.
"""

import random

import pytest

from plan_util import call, plan_of, tile_of

FRAG = 1536
BM, BN = 128, 256
SLOT_BYTES = 32 * 256 * 4 * 4


def check_gemm6(M_pad, N, K, M_out, N_out, k_split=0):
    """The launch in large tiles (by the library's own division for k_split 0, an operand being off its alignment)."""
    plan = plan_of(call("plain", M_out, K, N, 0, False, k_split=k_split, aligned=False))
    assert not plan.few_rows
    nblocks, kgroups, kparts = (N + BN - 1) // BN, K // 64, plan.kparts
    ntiles = (plan.full_blocks + plan.half_blocks) * nblocks
    act_bytes = M_pad * K * 3 // 4
    wgt_bytes = nblocks * BN * K * 3 // 4
    wsc_bytes = nblocks * kgroups * 2048
    asc_bytes = kgroups * M_pad * 2
    part_bytes = ntiles * kparts * SLOT_BYTES if kparts > 1 else 0
    total = ntiles * kparts
    seen = {}
    for bid in range(total):
        t = tile_of(plan, N, bid)
        m0, nb, part, MT = t.row, t.column_block, t.part, t.rows // 64
        assert 0 <= m0 and m0 + t.rows <= M_pad and 0 <= nb < nblocks and 0 <= part < kparts, (bid, m0, nb)
        mb, slab0 = m0 // 128, m0 % 128 // 32
        gb = kgroups * part // kparts
        ng = kgroups * (part + 1) // kparts - gb
        assert ng >= 1
        assert (m0, nb, part) not in seen
        seen[(m0, nb, part)] = True
        # the copy schedule: which k-groups get their weights (W) and the rest (R) requested
        w_req, r_req = [0], [0]
        if ng > 1:
            w_req.append(1)
            r_req.append(1)
        if ng > 2:
            w_req.append(2)
        l = 0
        while l + 3 < ng:  # MODE 2
            r_req.append(l + 2)
            w_req.append(l + 3)
            l += 1
        if l + 2 < ng:  # MODE 1
            r_req.append(l + 2)
            l += 1
        assert w_req == list(range(ng)) and r_req == list(range(ng)), (ng, w_req, r_req)
        for wave in range(4):
            for g in (0, ng // 2, ng - 1):  # (addresses grow with g)
                # three 1 KB weight chunks, 16 bytes per lane
                src_w = (nb * kgroups + gb + g) * 8 * FRAG + wave * 3072
                assert src_w + 2048 + 63 * 16 + 16 <= wgt_bytes
                act0 = (mb * kgroups + gb + g) * 4 * FRAG + slab0 * FRAG
                ws0 = (nb * kgroups + gb + g) * 2048
                as0 = ((gb + g) * M_pad + m0) * 2
                if MT == 2:
                    assert act0 + wave * 1024 + 1024 <= act_bytes
                    if wave < 2:
                        assert act0 + (4 + wave) * 1024 + 1024 <= act_bytes
                    else:
                        assert ws0 + (wave - 2) * 1024 + 1024 <= wsc_bytes
                    assert as0 + 63 * 4 + 4 <= asc_bytes
                elif wave < 3:  # two fragments are three chunks; the scales of 64 rows, eight times over
                    assert act0 + wave * 1024 + 1024 <= act0 + 2 * FRAG and act0 + 2 * FRAG <= act_bytes
                    assert as0 + 7 * 16 + 16 == as0 + 64 * 2 <= asc_bytes
                else:
                    assert ws0 + 1024 + 1024 <= wsc_bytes
        if kparts > 1:
            slot = (t.tile * kparts + part) * SLOT_BYTES
            assert slot + ((7 * 4 + 3) * 256 + 255) * 16 + 16 <= part_bytes
            assert t.tile * 4 + 4 <= ntiles * 4  # arrival counter
        # output stores: rows below M_out, 16-byte pieces below N_out
        for wm in range(2):
            for wn in range(2):
                for mt in range(MT):
                    for rr in (0, 31):
                        for cc in (0, 120):
                            m, n = m0 + wm * 32 * MT + mt * 32 + rr, nb * BN + wn * 128 + cc
                            if m < M_out and n < N_out:
                                assert (m * N_out + n) * 2 + 16 <= M_out * N_out * 2
    assert len(seen) == total
    return kparts


def buffer_read(size, voff, soff, nbytes, memory):
    """A request that is meant to read: inside the descriptor's size by either check, and inside the memory behind its base."""
    assert 0 <= size < 1 << 31 and 0 <= voff and 0 <= soff < 1 << 31
    assert voff + soff + nbytes <= size <= memory


def buffer_skip(size, voff, soff):
    """A request that is meant to touch no memory: outside by either check, without a sum beyond 32 bits."""
    assert voff >= size and voff + soff < 1 << 32


def check_direct(M, K, N, fp4, shape, rows):
    """The operands of the few-rows kernel (csrc/gemm_direct_kernel.h) in tiles of 32 `shape` rows."""
    M_pad, kgroups = (M + 255) // 256 * 256, K // 64
    MT, WN, KP = (1, 1, 4) if shape == 1 else (2, 1, 4) if fp4 else (2, 2, 2)
    NT, TILE = 4 // WN, 1024
    row_blocks = (rows + 32 * MT - 1) // (32 * MT)
    act_bytes, asc_bytes = (M_pad * K // 2, kgroups * M_pad * 4) if fp4 else (M_pad * K * 3 // 4, kgroups * M_pad * 2)
    padded = (N + 255) // 256 * 256  # (INT4 weights are stored in whole blocks of 256 columns)
    wgt_bytes, wsc_bytes = (N * K // 2, kgroups * N * 8) if fp4 else (padded * K * 3 // 4, padded // 256 * kgroups * 2048)
    total = row_blocks * (N // 128)
    seen = set()
    for bid in range(total):
        xcd, extra = bid % 8, total % 8
        v = xcd * (total // 8) + min(xcd, extra) + bid // 8
        nb, mb = divmod(v, row_blocks)
        seen.add((nb, mb))
        assert nb < N // 128 and (mb + 1) * 32 * MT <= M_pad
        f0 = mb * MT
        for kpart in range(KP):
            g_load = min(kpart, kgroups - 1)
            last = kpart + (kgroups - 1 - kpart) // KP * KP if kpart < kgroups else g_load  # the group the requests stop at
            assert last < kgroups and last + KP >= kgroups
            for g in {g_load, last}:
                for mt in range(MT):
                    if fp4:
                        assert ((f0 + mt) * kgroups + g) * TILE + 31 * 32 + 16 + 16 <= act_bytes
                        assert (g * M_pad + f0 * 32) * 4 + mt * 128 + 31 * 4 + 2 + 2 <= asc_bytes
                    else:
                        assert ((f0 + mt) // 4 * kgroups + g) * 4 * FRAG + (f0 + mt) % 4 * FRAG + 1024 + 63 * 8 + 8 <= act_bytes
                        assert (g * M_pad + f0 * 32) * 2 + mt * 64 + 31 * 2 + 2 <= asc_bytes
                for cw in range(WN):
                    for nt in range(NT):
                        if fp4:
                            # as buffers: size, lane's offset, scalar offset
                            s_lead, a_lead = (nb * 128 + cw * NT * 32) * 8, f0 * 32 * 4
                            buffer_read(NT * kgroups * TILE, 31 * 32 + 16, g * TILE + nt * kgroups * TILE, 16, wgt_bytes - (nb * 4 + cw * NT) * kgroups * TILE)
                            buffer_read(kgroups * N * 8 - s_lead, 31 * 8 + 4 + nt * 256, g * N * 8, 4, wsc_bytes - s_lead)
                            for mt in range(MT):
                                buffer_read(MT * kgroups * TILE, 31 * 32 + 16, g * TILE + mt * kgroups * TILE, 16, act_bytes - f0 * kgroups * TILE)
                                buffer_read(kgroups * M_pad * 4 - a_lead, 31 * 4 + 2 + mt * 128, g * M_pad * 4, 2, asc_bytes - a_lead)
                            assert ((nb * 4 + cw * NT) * kgroups + g) * TILE + nt * kgroups * TILE + 31 * 32 + 16 + 16 <= wgt_bytes
                            assert (g * N + nb * 128 + cw * NT * 32) * 8 + nt * 256 + 31 * 8 + 4 + 4 <= wsc_bytes
                        else:
                            assert (nb // 2 * kgroups + g) * 8 * FRAG + (nb % 2 * 4 + cw * NT + nt) * FRAG + 1024 + 63 * 8 + 8 <= wgt_bytes
                            assert (nb // 2 * kgroups + g) * 2048 + nb % 2 * 1024 + cw * NT * 256 + nt * 256 + 31 * 8 + 4 <= wsc_bytes
    assert len(seen) == total and rows <= row_blocks * 32 * MT


def sweep_shapes():
    """The distribution of the seeded sweep and of the randomized loop (test_gpu_shape_sweep.py), INT4 cases."""
    shapes = {(100, 3072, 768, 0), (100, 3072, 768, 3)}
    for seed in (1, 2, 3):
        rng = random.Random(seed)
        for _ in range(400):
            fp4 = rng.random() < 0.3
            M = rng.choice([1, 17, 100, 255, 256, 257, 300, 511, 640, 900, 1300])
            K = 128 * rng.randint(1, 9) if rng.random() < 0.7 else rng.choice([2048, 3072, 4096, 6144])
            N = 128 * rng.randint(1, 11)
            rng.choice([0, 16, 32, 32, 48, 64, 96, 128])
            rng.random(), rng.random(), rng.choice([1.0, 1.0, 0.5, 1.7]) if not fp4 else None, rng.random()
            ks = rng.choice([None, None, None, 1, 2, 3, 5]) if not fp4 else rng.choice([None, None, 1, 2])
            if not fp4:
                shapes.add((M, K, N, ks or 0))
    return sorted(shapes)


def test_gemm6_addresses_stay_inside_their_buffers():
    shapes = sweep_shapes()
    assert (100, 3072, 768, 0) in shapes
    for M, K, N, ks in shapes:
        M_pad = (M + 255) // 256 * 256
        check_gemm6(M_pad, N, K, M, N, ks)
    # the case that faulted: six tiles, by the library's own choice split in three parts then and, in large tiles, in four now
    assert check_gemm6(256, 768, 3072, 100, 768, 0) == 4
    assert check_gemm6(256, 768, 3072, 100, 768, 3) == 3


def test_gemm6_addresses_large_shapes():
    for M_pad, N, K in ((4608, 12288, 3072), (4608, 3072, 12288), (4608, 9216, 3072), (256, 3072, 3072)):
        check_gemm6(M_pad, N, K, M_pad, N, 0)


@pytest.mark.parametrize("fp4", [False, True])
def test_few_rows_addresses_stay_inside_their_buffers(fp4):
    for M, K, N, _ in sweep_shapes()[::3] + [(1, 128, 128, 0), (4608, 3072, 3072, 0), (1157, 12288, 3072, 0)]:
        M_pad = (M + 255) // 256 * 256
        for shape in (1, 2):
            for rows in {M, M_pad}:
                check_direct(M, K, N, fp4, shape, rows)


def test_projecting_workgroups_read_inside_proj_down():
    """csrc/quantize.hip, project_rows: rank tile rt of step i of chunk c is the KB behind ((4 c + i) R / 16 + rt) KB; a second rank
    tile beyond the rank repeats the first.  (Its rows are read as the quantize kernel's with 16 rows are.)"""
    for K in (128, 1152, 12288):
        for R in (16, 48, 80, 1024):
            RT = R // 16
            for RTW in (1, 2):
                for rt0 in range(0, RT, RTW):
                    rt1 = rt0 + 1 if rt0 + 1 < RT else rt0
                    for rt in (rt0, rt1):
                        assert ((K // 128 - 1) * 4 + 3) * RT * 1024 + rt * 1024 + 63 * 16 + 16 <= K * R * 2


@pytest.mark.parametrize("glu", [False, True])
def test_quantize_row_buffer_cuts_exactly_at_the_last_row(glu):
    """The kernel reads x through a raw buffer whose size (num_records) ends with the workgroup's last valid row, and
    carries the 128-column chunk in the scalar offset.  Whether the hardware's range check counts the scalar offset or not, a
    lane reads memory if and only if its row is valid (and the chunk exists: past the last chunk the kernel sets bit 31
    of the lane offset)."""
    XW = 2 if glu else 1
    PPR, RPI = 16 * XW, 64 // (16 * XW)
    for K in (128, 256, 1152, 3072, 12288):
        ld = XW * K
        nchunks = K // 128
        for MT in (1, 2):
            for rows_valid in (0, 1, 5, 15, 16, 17, 31, 32):
                rv = min(rows_valid, 16 * MT)
                num_records = rv * ld * 2
                for c in (0, nchunks - 1, nchunks, nchunks + 3):
                    beyond = 0 if c < nchunks else 0x80000000
                    soffset = c * 256 * XW
                    for mt in range(MT):
                        for i in range(4 * XW):
                            for lane in range(64):
                                row = 16 * mt + RPI * i + lane // PPR
                                voff = ((lane // PPR) * ld * 2 + (lane % PPR) * 16) | beyond
                                voff += (16 * mt + RPI * i) * ld * 2
                                in_range = voff + 16 <= num_records
                                assert in_range == (row < rv and c < nchunks), (K, MT, rows_valid, c, mt, i, lane)
                                assert in_range == (voff + soffset + 16 <= num_records) and voff + soffset < 1 << 32
                                if in_range:  # the bytes a lane in range touches belong to its row and chunk
                                    first = voff + soffset
                                    assert row * ld * 2 + c * 256 * XW <= first and first + 16 <= row * ld * 2 + (c + 1) * 256 * XW


def test_quantize_store_addresses():
    for M, K, R in ((1, 128, 0), (100, 3072, 32), (257, 1152, 160), (300, 256, 1024), (4608, 3072, 32)):
        M_pad = (M + 255) // 256 * 256
        kgroups = K // 64
        act_bytes, asc_elems, lora_elems = M_pad * K * 3 // 4, kgroups * M_pad, M_pad * R
        for row in (0, 31, 127, 128, M_pad - 1):
            for c in (0, K // 128 - 1):
                for q in range(4):
                    g = 2 * c + (q >> 1)
                    frag = ((row // 128 * kgroups + g) * 4 + (row % 128) // 32) * FRAG
                    slot = row % 32 + 32 * (q & 1)
                    assert frag + slot * 16 + 16 <= act_bytes and frag + 1024 + slot * 8 + 8 <= act_bytes
                    assert g * M_pad + row < asc_elems
            if R:
                for rt_base in range(0, R // 16, 8):
                    rts = min(R // 16 - rt_base, 8)
                    for rank in (0, 16 * rts - 1):
                        assert row * R + 16 * rt_base + rank < lora_elems


@pytest.mark.parametrize("R", [16, 32, 48, 128, 144, 256, 1024])
def test_low_rank_operands_stay_inside_their_buffers(R):
    """The operands of the up projection, lora_act [M_pad][R] fp32 and lora_up [N][R] bf16.  INT4 (csrc/gemm6_kernel.h, request_chunk):
    chunks of 32 ranks by asynchronous copies, 64 bytes of each of 256 columns and 128 bytes of each of 64 MT rows; columns beyond N
    repeat the last, half a chunk repeats its 16 ranks.  NVFP4 (csrc/gemm_kernel.h, request): windows of 128 ranks, 32 at a time."""
    steps = R // 16
    for N in (128, 256, 384, 640):
        for n0 in range(0, N, 256):
            for c in range((steps + 1) // 2):
                half = steps - 2 * c < 2
                pieces, places = set(), {}
                for wave in range(4):
                    for i in range(4):
                        for lane in range(64):
                            row = (wave * 4 + i) * 16 + (lane >> 2)
                            piece = (lane & 3) ^ ((row >> 2) & 3)
                            column = n0 + (row if n0 + row < N else N - 1 - n0)
                            first = column * R * 2 + c * 64 + (piece & 1 if half else piece) * 16
                            assert column * R * 2 <= first and first + 16 <= (column + 1) * R * 2 <= N * R * 2
                            place = (wave * 4 + i) * 1024 + lane * 16
                            assert place not in places and place == row * 64 + (piece ^ ((row >> 2) & 3)) * 16
                            places[place] = (row, piece)
                            pieces.add((row, piece))
                assert len(pieces) == 256 * 4
    for MT in (1, 2):
        for M_pad in (256, 512):
            for m0 in range(0, M_pad, 64 * MT):
                for c in range((steps + 1) // 2):
                    half = steps - 2 * c < 2
                    pieces = set()
                    for wave in range(4):
                        for i in range(2 * MT):
                            for lane in range(64):
                                row = (wave * 2 * MT + i) * 8 + (lane >> 3)
                                piece = (lane & 7) ^ ((row >> 1) & 7)
                                first = (m0 + row) * R * 4 + c * 128 + (piece & 3 if half else piece) * 16
                                assert first + 16 <= (m0 + row + 1) * R * 4 <= M_pad * R * 4
                                assert (wave * 2 * MT + i) * 1024 + lane * 16 == row * 128 + (piece ^ ((row >> 1) & 7)) * 16
                                pieces.add((row, piece))
                    assert len(pieces) == 64 * MT * 8
    for first in range(0, steps, 8):
        window, seen = min(steps - first, 8), set()
        for c in range((window + 1) // 2):
            for lane in range(64):
                step = first + 2 * c + (1 if lane & 4 and 2 * c + 1 < window else 0)
                up_step = first + 2 * c + (1 if lane & 2 and 2 * c + 1 < window else 0)
                assert 16 * step + (lane & 3) * 4 + 4 <= R and 16 * up_step + (lane & 1) * 8 + 8 <= R
                for place, limit in ((2 * c + ((lane & 4) >> 2), "act"), (2 * c + ((lane & 2) >> 1), "up")):
                    if place < window:  # (what is written to LDS is what was requested)
                        assert first + place == (step if limit == "act" else up_step)
                        seen.add((limit, place))
        assert seen == {(name, place) for name in ("act", "up") for place in range(window)}


@pytest.mark.parametrize("N,K,ncu", [(16, 640, 256), (20, 1088, 256), (4092, 640, 256), (9220, 640, 256), (18432, 3072, 256), (24572, 640, 256), (20480, 4096, 304),
                                     ((1 << 24) - 4, 4096, 256)])
def test_awq_shares_read_inside_their_buffers(N, K, ncu):
    """The AWQ GEMV with one workgroup per compute unit: the shares cover the channels once; a lane whose channel is the share's reads its
    codes, scale and zero, any other (the share's last tile, the tiles requested ahead) nothing."""
    kblocks, BATCH, AHEAD = K // 64, 6, 2
    assert kblocks * N < 1 << 30  # (the launcher's condition)
    spw = ((K + 127) // 128 + 7) // 8
    grid = min((N + 15) // 16, ncu)
    share, more, covered = N // 4 // grid, N // 4 % grid, 0
    for wg in range(grid):
        begin = 4 * (wg * share + min(wg, more))
        end = begin + 4 * (share + (1 if wg < more else 0))
        assert begin == covered
        covered = end
        if wg not in (0, 1, more - 1, more, grid - 2, grid - 1):
            continue
        tiles = (end - begin + 15) // 16
        requested = list(range(AHEAD))
        for t0 in range(0, tiles, BATCH):
            requested += [t0 + i + AHEAD for i in range(min(tiles - t0, BATCH))]
        assert set(range(tiles)) <= set(requested)
        w_size, s_size = (end - begin) // 4 * kblocks * 128, kblocks * N * 2
        assert w_size < 1 << 31 and s_size < 1 << 31
        for t in {0, 1, tiles - 1, tiles, tiles + 1} & set(requested):
            for n in range(16):
                for j in (0, spw - 1):
                    for wave in (0, 7):
                        for kb in range(4):
                            cb = (wave + 8 * j) * 2 + (kb >> 1)
                            block = min(cb, kblocks - 1)
                            w_off = (n >> 2) * kblocks * 128 + (n & 3) * 32 + (kb & 1) * 16 + block * 128
                            s_off = block * N * 2 + n * 2
                            wt, st = t * kblocks * 512, (begin + 16 * t) * 2
                            channel = begin + 16 * t + n
                            if channel < end:
                                buffer_read(w_size, w_off, wt, 16, N // 4 * kblocks * 128 - begin // 4 * kblocks * 128)
                                buffer_read(s_size, s_off, st, 2, s_size)
                                assert begin // 4 * kblocks * 128 + w_off + wt == ((channel // 4 * kblocks + block) * 4 + channel % 4) * 32 + (kb & 1) * 16
                                assert (s_off + st) // 2 == block * N + channel
                            else:
                                buffer_skip(w_size, w_off | 0x80000000, wt)
                                buffer_skip(s_size, s_off | 0x80000000, st)
    assert covered == N
