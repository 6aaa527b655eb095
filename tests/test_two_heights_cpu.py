"""How NVFP4 few-rows launches of 64 x 128 tiles divide their rows into blocks of 64 and 32 rows (csrc/gemm.hip, ``few_rows_heights``) and number the tiles
(csrc/gemm_direct_kernel.h, ``gemm_direct_kernel``)."""

import random

import pytest

from plan_util import call, plan_of


def tile_of(block: int, total: int) -> int:  # (as in the kernel)
    xcd, extra = block % 8, total % 8
    return xcd * (total // 8) + min(xcd, extra) + block // 8


def tiles(full: int, half: int, columns: int):
    """(first row, rows, column block) of every workgroup, as the kernel works them out."""
    whole, total = full * columns, (full + half) * columns
    for block in range(total):
        if block < whole:
            nb, mb = divmod(tile_of(block, whole), full)
            yield mb * 64, 64, nb
        else:
            nb, mb = divmod(tile_of(block - whole, total - whole), half)
            yield full * 64 + mb * 32, 32, nb


@pytest.mark.parametrize("full,half,columns", [(1, 1, 1), (3, 4, 72), (16, 5, 96), (5, 1, 7), (2, 0, 9)])
def test_every_tile_once(full, half, columns):
    got = sorted(tiles(full, half, columns))
    want = [(64 * i, 64, n) for i in range(full) for n in range(columns)] + [(64 * full + 32 * i, 32, n) for i in range(half) for n in range(columns)]
    assert got == want


def test_rows_are_covered_inside_the_padded_tensor():
    """Against the busiest compute unit's tiles, counted one by one: never more than with 64-row tiles alone."""
    rng, mixed = random.Random(1), 0
    for _ in range(4000):
        kind, M, K, N = rng.choice(["plain", "silu", "rope", "litela"]), rng.randint(1, 3000), 128 * rng.randint(1, 30), 384 * rng.randint(1, 40)
        if kind == "litela":
            M = (M + 255) // 256 * 256
        ncu = rng.choice([256, 256, 304, 64])
        p = plan_of(call(kind, M, K, N, 32, True), compute_units=ncu)
        if (p.few_rows, p.columns) != (2, 128):
            assert p.full_blocks == 0
            continue
        units, nb = (M + 31) // 32, N // 128
        half = max(units - 2 * p.full_blocks, 0)
        assert p.row_blocks == (M + 63) // 64 and 0 < p.full_blocks <= p.row_blocks and M <= 64 * p.full_blocks + 32 * half <= (M + 255) // 256 * 256
        load = [0.0] * ncu
        for cost, n in ((1.0, p.full_blocks * nb), (0.68, half * nb)):
            for _ in range(n):  # the emptiest one takes the next tile
                i = min(range(ncu), key=load.__getitem__) if half else 0
                load[i] += cost if half else 0.0
        if half:
            mixed += 1
            assert max(load) <= 0.985 * -(-p.row_blocks * nb // ncu) + 1e-9
    assert mixed > 100


@pytest.mark.parametrize("kind,M,K,N,want", [
    ("rope", 505, 3072, 9216, 7), ("rope", 300, 3072, 9216, 3), ("silu", 201, 2688, 15744, 4), ("plain", 2300, 3072, 3072, 32), ("rope", 1200, 3072, 9216, 17),
    ("split", 17, 3968, 11904, 4), ("plain", 800, 3072, 3072, 10), ("plain", 405, 2944, 5120, 6), ("split", 2422, 1920, 5760, 39),  # (the last three in other tiles but for those of 32 rows)
])
def test_blocks_of_64_rows(kind, M, K, N, want):
    p = plan_of(call(kind, M, K, N, 32, True))
    assert (p.few_rows, p.columns, p.full_blocks) == (2, 128, want), p
    assert plan_of(call(kind, M, K, N, 32, False)).few_rows * plan_of(call(kind, M, K, N, 32, False)).full_blocks == 0
    assert plan_of(call("next", 1157, 3072, 12288, 32, True, with_out=False), rows=1157).full_blocks == 16


# No two heights where 32-row tiles alone are two per compute unit at most (465 to 507 of them in the first seven, 513 and 520 in the others), whichever model chooses the tile.
@pytest.mark.parametrize("kind,M,K,N,R,mt", [
    ("silu", 67, 2944, 19840, 16, 1), ("silu", 66, 7424, 19072, 32, 1), ("next", 65, 6272, 18176, 64, 1), ("plain", 68, 12928, 19584, 64, 1), ("silu", 587, 13568, 3328, 32, 1),
    ("next", 1227, 3584, 1664, 32, 1), ("plain", 513, 11904, 3712, 0, 1), ("silu", 587, 13568, 3456, 32, 2), ("next", 1250, 3584, 1664, 32, 2),
])
def test_two_heights_from_three_32_row_tiles_on(kind, M, K, N, R, mt):
    p = plan_of(call(kind, M, K, N, R, True, with_out=kind != "next", R_down=R), rows=M if kind == "next" else 0)
    assert (p.few_rows, p.columns) == (mt, 128), p


# Ranks above 32 cost the few-rows kernel less (their operands come through LDS): on either side of the line to whole large tiles.
@pytest.mark.parametrize("kind,M,K,N,R,few", [
    ("split", 3235, 1408, 4224, 80, 2), ("rope", 6509, 1536, 4608, 64, 2), ("silu", 2881, 1408, 18304, 128, 2), ("plain", 4709, 1408, 3328, 128, 0), ("plain", 4608, 3072, 21504, 32, 0),
])
def test_few_rows_or_large_tiles_at_higher_ranks(kind, M, K, N, R, few):
    assert plan_of(call(kind, M, K, N, R, True)).few_rows == few


# ... and short rows less so (the first seven were up to 28 percent slower than in large tiles); ranks 0 and 16 at K = 128 by 64-row tiles alone (the next three, 17 percent).
@pytest.mark.parametrize("kind,M,K,N,R,few", [
    ("plain", 15370, 128, 1920, 80, 0), ("rope", 10352, 384, 3072, 64, 0), ("litela", 10240, 128, 13056, 112, 0), ("rope", 13290, 384, 6912, 112, 0), ("plain", 17195, 512, 1792, 80, 0),
    ("plain", 8637, 384, 3584, 96, 0), ("rope", 8151, 128, 3840, 48, 0), ("plain", 4481, 128, 3456, 0, 0), ("plain", 11853, 128, 1280, 0, 0), ("plain", 2333, 128, 12544, 16, 0),
    ("plain", 15370, 1152, 1920, 80, 2), ("rope", 10352, 1536, 3072, 64, 2), ("litela", 3072, 128, 13056, 112, 2), ("silu", 11853, 256, 1280, 16, 2), ("plain", 12799, 128, 896, 32, 2),
])
def test_few_rows_or_large_tiles_at_short_rows(kind, M, K, N, R, few):
    assert plan_of(call(kind, M, K, N, R, True)).few_rows == few
