"""The tile numbering of the INT4 GEMM (csrc/gemm6_kernel.h, gemm6_kernel) restated on the CPU: every tile of a launch is
taken by exactly one workgroup, whatever the numbers of 128-row and 64-row blocks, and the rows a launch divides into them
(csrc/gemm.hip, choose_row_blocks) are covered without leaving the padded tensor."""

import pytest


def band_height(blocks, most):
    bands = (blocks + most - 1) // most
    return (blocks + bands - 1) // bands if bands else 1


def tile_of(block_idx, total, full_blocks, half_blocks, nblocks, kparts=1):
    """(first row, column block, part, rows) of a workgroup."""
    full = full_blocks * nblocks * kparts
    xcd, j = block_idx % 8, block_idx // 8
    first = xcd * (full // 8) + min(xcd, full % 8)
    count = full // 8 + (xcd < full % 8)
    whole = j < count
    v = first + j if whole else xcd * (total // 8) + min(xcd, total % 8) - first + (j - count)
    tile, part = divmod(v, kparts) if whole else (v, 0)
    blocks = full_blocks if whole else half_blocks
    BAND = band_height(full_blocks, 10) if whole else band_height(half_blocks, 20)
    band, in_band = divmod(tile, BAND * nblocks)
    rows = min(BAND, blocks - band * BAND)
    mb, nb = band * BAND + in_band % rows, in_band // rows
    return (mb * 128, nb, part, 128) if whole else (full_blocks * 128 + mb * 64, nb, 0, 64)


def unit_time(whole, half):
    pairs = 1.55 * (whole // 2)
    if whole % 2 == 0:
        return pairs + 0.9 * (half // 2) + 0.7 * (half % 2)
    return pairs + (1.0 if half == 0 else 1.1 if half == 1 else 2.0 + 0.25 * (half - 2))


def launch_time(whole, half, ncu):
    q, more = divmod(whole, ncu)
    fewer, h0, h1 = ncu - more, 0, 0
    t = unit_time(q + 1, 0) if more else unit_time(q, 0)
    while True:
        while unit_time(q, h0 + 1) <= t:
            h0 += 1
        while unit_time(q + 1, h1 + 1) <= t:
            h1 += 1
        if h0 * fewer + h1 * more >= half:
            return t
        t0, t1 = unit_time(q, h0 + 1), unit_time(q + 1, h1 + 1)
        t = t1 if more and t1 < t0 else t0


def choose_row_blocks(rows, nblocks, ncu=256):
    """csrc/gemm.hip::choose_row_blocks: (128-row blocks, 64-row blocks, modelled time in tiles)"""
    units = (rows + 63) // 64
    full = (units + 1) // 2
    tiles = full * nblocks
    q = (tiles - 1) // ncu
    best = (full, 0, launch_time(tiles, 0, ncu))
    to_beat = 0.96 * best[2]
    for f in [q * ncu // nblocks] + ([(q - 1) * ncu // nblocks] if q else []) + ([0] if tiles <= 2 * ncu else []):
        f = min(f, units // 2)
        h = units - 2 * f
        if h and (t := launch_time(f * nblocks, h * nblocks, ncu)) <= to_beat:
            to_beat, best = t, (f, h, t)
    return best


@pytest.mark.parametrize("nblocks", [1, 3, 12, 27, 36, 48])
def test_every_tile_once(nblocks):
    for full in (0, 1, 2, 7, 9, 10, 11, 36):
        for half in (0, 1, 2, 5, 20, 21):
            for kparts in ((1, 3) if half == 0 else (1,)):
                total = (full * kparts + half) * nblocks
                got = [tile_of(b, total, full, half, nblocks, kparts) for b in range(total)]
                want = {(mb * 128, nb, part, 128) for mb in range(full) for nb in range(nblocks) for part in range(kparts)}
                want |= {(full * 128 + mb * 64, nb, 0, 64) for mb in range(half) for nb in range(nblocks)}
                assert len(set(got)) == total and set(got) == want, (full, half, kparts)


def test_rows_are_covered_inside_the_padded_tensor():
    for nblocks in (1, 4, 12, 27, 36, 48, 84):
        for rows in [*range(1, 2200, 37), 4096, 4608, 9216, 18432, 18433]:
            f, h, t = choose_row_blocks(rows, nblocks)
            m_pad = (rows + 255) // 256 * 256
            assert rows <= f * 128 + h * 64 <= m_pad and f * 128 + h * 64 - rows < 128
            assert t <= launch_time((rows + 127) // 128 * nblocks, 0, 256)  # never modelled slower than whole tiles alone
