"""The tiles of few-rows GEMM launches, asked of the library (csrc/internal_api.h): every tile once, inside the padded rows, and the operands of both heights inside
their buffers (by the address model's range checks)."""

import ctypes
import random

from nunchaku_amd import _native as nv
from plan_util import Tile, call, plan_of
from test_address_model import buffer_read

TILE = 1024


def tiles_of(plan, N):
    lib, N, block, total = nv.lib(), ctypes.c_int64(N), 0, 1
    while block < total:
        t = Tile()
        total = lib.svdq_gemm_few_rows_tile(ctypes.byref(plan), N, block, ctypes.byref(t))
        yield t
        block += 1


def launches(n):
    rng = random.Random(7)
    for _ in range(n):
        kind, M, K, N = rng.choice(["plain", "silu", "next", "rope", "litela"]), rng.choice([1, 31, 64, 65, rng.randint(66, 2500)]), 128 * rng.randint(1, 12), 384 * rng.randint(1, 24)
        if kind == "litela":
            M = (M + 255) // 256 * 256
        yield kind, M, K, N, rng.random() < 0.3
    yield from [("rope", 505, 3072, 9216, False), ("next", 1157, 3072, 12288, False), ("plain", 800, 3072, 3072, False), ("plain", 929, 1024, 4608, False), ("plain", 40, 256, 128, True)]


def test_every_tile_once_and_inside_its_buffers():
    mixed = 0
    for kind, M, K, N, int4 in launches(500):
        p = plan_of(call(kind, M, K, N, 32, not int4, with_out=kind != "next"), rows=M if kind == "next" else 0)
        if not p.few_rows:
            continue
        M_pad, columns, kgroups = (M + 255) // 256 * 256, p.columns, K // 64
        mixed += p.low_blocks > 0
        # (first row, rows, first column); the rows that the blocks cover without a gap or an overlap
        got = [(t.row, t.rows, t.column_block * columns) for t in tiles_of(p, N)]
        blocks = sorted({(r, h) for r, h, _ in got})
        assert len(got) == len(set(got)) == len(blocks) * (N // columns) and {c for _, _, c in got} == set(range(0, N, columns))
        assert [r for r, _ in blocks] == [sum(h for _, h in blocks[:i]) for i in range(len(blocks))]
        covered = blocks[-1][0] + blocks[-1][1]
        assert M <= covered <= M_pad and covered - M < blocks[-1][1], p
        assert [h for _, h in blocks] == ([64] * p.full_blocks + [32] * p.low_blocks if p.full_blocks else [32 * p.few_rows] * p.row_blocks), p
        if int4 or columns < 128:
            continue
        for row, rows, col in {(r, h, c) for r, h, c in got if c in (0, N - 128)}:
            MT, nb, f0 = rows // 32, col // 128, row // 32
            s_lead, a_lead = col * 8, row * 4
            for g in {0, kgroups - 1}:
                buffer_read(4 * kgroups * TILE, 31 * 32 + 16, g * TILE + 3 * kgroups * TILE, 16, N * K // 2 - nb * 4 * kgroups * TILE)
                buffer_read(kgroups * N * 8 - s_lead, 31 * 8 + 4 + 3 * 256, g * N * 8, 4, kgroups * N * 8 - s_lead)
                buffer_read(MT * kgroups * TILE, 31 * 32 + 16, g * TILE + (MT - 1) * kgroups * TILE, 16, M_pad * K // 2 - f0 * kgroups * TILE)
                buffer_read(kgroups * M_pad * 4 - a_lead, 31 * 4 + 2 + (MT - 1) * 128, g * M_pad * 4, 2, kgroups * M_pad * 4 - a_lead)
    assert mixed >= 20
