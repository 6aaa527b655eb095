"""The tiles of few-rows GEMM launches and the asynchronous copies of their low-rank operands, asked of the library (csrc/internal_api.h): every tile once, inside
the padded rows, the operands of both heights inside their buffers (by the address model's range checks), every copy inside its operand and its place in LDS, and
behind every place that a multiplying lane reads the bytes that it wants."""

import ctypes
import random

import pytest

from nunchaku_amd import _native as nv
from plan_util import Tile, call, plan_of
from test_address_model import buffer_read

TILE = 1024


class LowRank(ctypes.Structure):
    """Mirror of ``svdq_gemm_low_rank``."""

    _fields_ = [(n, ctypes.c_int32) for n in ("first", "end", "steps", "chunk", "act", "up_requests", "act_requests")]


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


@pytest.mark.parametrize("form,rows", [(0, 64), (1, 32), (2, 64)])
def test_copies_of_the_low_rank_operands(form, rows):
    lib = nv.lib()
    lib.svdq_gemm_low_rank_copied.restype = ctypes.c_int64

    def copied(act, first, *where):
        return lib.svdq_gemm_low_rank_copied(act, ctypes.c_int64(first), *where)

    for R in [*range(16, 273, 16), 496, 1024]:
        for three in (0, 1) if form == 0 else (0,):
            c = LowRank()
            lib.svdq_gemm_low_rank_of(form, R, three, ctypes.byref(c))
            chunks = (c.steps + 1) // 2
            assert 0 < c.steps <= R // 16 and c.first + chunks * c.chunk <= c.end <= (160 * 1024 // (3 if three else 2))
            for act, index, size, pieces, requests, base in ((0, 128, 2, 4, c.up_requests, 0), (1, rows, 4, 8, c.act_requests, c.act)):
                # a request's lane puts 16 bytes behind those of the lane before it; a column's (row's) 32 ranks are `pieces` of them
                assert requests * 64 == index * pieces and base + requests * 1024 <= (c.act if not act else c.chunk)
                total = (3 * index + index) * R * size  # (the operand ends with the tile: it starts at its column or row 3 index)
                for chunk in {0, chunks - 1}:
                    source = {}
                    for request in range(requests):
                        for lane in range(64):
                            at = copied(act, 3 * index, R, chunk, request, lane)
                            assert at % 16 == 0 and 3 * index * R * size <= at and at + 16 <= total, (form, R, act, chunk, request, lane)
                            source[request * 1024 + lane * 16] = at
                    left = min(2, c.steps - 2 * chunk) * pieces // 2
                    places = set()
                    for i in range(index):
                        for piece in range(left):
                            place = lib.svdq_gemm_low_rank_place(act, i, piece)
                            places.add(place)
                            assert source[place] == (3 * index + i) * R * size + chunk * 32 * size + piece * 16, (form, R, act, chunk, i, piece)
                    assert len(places) == index * left
