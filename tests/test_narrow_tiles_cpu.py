"""The few-rows GEMM's tiles with the plain epilogue (csrc/gemm.hip, ``plain_tile``; csrc/gemm_narrow_variant.hip) on the CPU: which one
a launch takes, that no operand is read outside its buffer, and that the kernels keep out of scratch memory."""

import re

import pytest

from plan_util import call, plan_of
from test_address_model import FRAG, buffer_read
from test_build_guard import compiled  # noqa: F401  (the fixture)


# (shape, the tile on 256 compute units; the same for both precisions)
@pytest.mark.parametrize("M,K,N,want", [
    (16, 1024, 1024, (32, 32)), (64, 3072, 3072, (32, 32)), (64, 12288, 3072, (32, 32)), (32, 3072, 12288, (32, 64)), (128, 3072, 3072, (64, 32)),
    (256, 3072, 3072, (64, 64)), (300, 3072, 3072, (64, 64)), (256, 12288, 3072, (64, 64)), (89, 2432, 20480, (32, 128)), (1157, 12288, 3072, (64, 128)),
])
@pytest.mark.parametrize("fp4", [False, True])
def test_the_tile_of_a_launch(M, K, N, want, fp4):
    p = plan_of(call("plain", M, K, N, 32, fp4))
    assert (32 * p.few_rows, p.columns) == want and p.shared_rows == ((M, fp4) == (1157, False)), p
    assert p.row_blocks == (M + want[0] - 1) // want[0], p


# Launches whose narrow tiles the INT4 model takes for faster than the 64 x 128 ones, which they are not: short rows and few columns, several tiles
# per compute unit; and ones where a tile of another height than that of the better one of 128 columns is the fastest.
@pytest.mark.parametrize("M,K,N,fp4,want", [
    (125, 128, 11392, False, (64, 128)), (500, 128, 2176, False, (64, 128)), (5494, 2560, 256, False, (64, 128)), (556, 2944, 4096, False, (64, 64)),
    (297, 1280, 3456, True, (32, 64)), (788, 4224, 7680, True, (64, 128)), (261, 1280, 21376, True, (64, 128)), (5041, 8448, 512, True, (64, 128)),
])
def test_narrow_tiles_only_where_they_are_faster(M, K, N, fp4, want):
    p = plan_of(call("plain", M, K, N, 32, fp4))
    assert (32 * p.few_rows, p.columns) == want, p


def check_addresses(M, K, N, fp4, MT, NC):
    """The requests of the first and the last k-group of every wave (four of them split K) for every tile of a launch."""
    M_pad, kgroups, TILE = (M + 255) // 256 * 256, K // 64, 1024
    row_blocks, column_blocks = (M + 32 * MT - 1) // (32 * MT), N // (32 * NC)
    act_bytes, asc_bytes = (M_pad * K // 2, kgroups * M_pad * 4) if fp4 else (M_pad * K * 3 // 4, kgroups * M_pad * 2)
    padded = (N + 255) // 256 * 256  # (INT4 weights are stored in whole blocks of 256 columns)
    wgt_bytes, wsc_bytes = (N * K // 2, kgroups * N * 8) if fp4 else (padded * K * 3 // 4, padded // 256 * kgroups * 2048)
    total, seen = row_blocks * column_blocks, set()
    for bid in range(total):
        xcd, extra = bid % 8, total % 8
        nb, mb = divmod(xcd * (total // 8) + min(xcd, extra) + bid // 8, row_blocks)
        seen.add((nb, mb))
        f0 = mb * MT
        assert nb < column_blocks and (f0 + MT) * 32 <= M_pad
        for g in {min(k, kgroups - 1) for k in range(4)} | {kgroups - 1, max(kgroups - 4, 0)}:
            for mt in range(MT):
                if fp4:
                    a_lead = f0 * 32 * 4
                    buffer_read(MT * kgroups * TILE, 31 * 32 + 16, g * TILE + mt * kgroups * TILE, 16, act_bytes - f0 * kgroups * TILE)
                    buffer_read(kgroups * M_pad * 4 - a_lead, 31 * 4 + 2 + mt * 128, g * M_pad * 4, 2, asc_bytes - a_lead)
                else:
                    assert ((f0 + mt) // 4 * kgroups + g) * 4 * FRAG + (f0 + mt) % 4 * FRAG + 1024 + 63 * 8 + 8 <= act_bytes
                    assert (g * M_pad + f0 * 32) * 2 + mt * 64 + 31 * 2 + 2 <= asc_bytes
            for nt in range(NC):
                if fp4:
                    s_lead = nb * 32 * NC * 8
                    buffer_read(NC * kgroups * TILE, 31 * 32 + 16, g * TILE + nt * kgroups * TILE, 16, wgt_bytes - nb * NC * kgroups * TILE)
                    buffer_read(kgroups * N * 8 - s_lead, 31 * 8 + 4 + nt * 256, g * N * 8, 4, wsc_bytes - s_lead)
                else:
                    block, tile = divmod(nb * NC + nt, 8)
                    assert divmod(nb, 8 // NC) == (block, (tile - nt) // NC)  # as the kernel has it
                    assert (block * kgroups + g) * 8 * FRAG + tile * FRAG + 1024 + 63 * 8 + 8 <= wgt_bytes
                    assert (block * kgroups + g) * 2048 + tile * 256 + 31 * 8 + 4 <= wsc_bytes
    assert len(seen) == total


@pytest.mark.parametrize("fp4", [False, True])
def test_addresses_stay_inside_their_buffers(fp4):
    for M, K, N in ((1, 128, 128), (33, 640, 384), (100, 3072, 768), (256, 3072, 3072), (300, 256, 1152), (769, 192 * 2, 640)):
        for MT, NC in ((1, 1), (1, 2), (2, 1), (2, 2)):
            check_addresses(M, K, N, fp4, MT, NC)


@pytest.mark.parametrize("variant", [0, 1])
def test_narrow_tiles_fit_their_registers(compiled, variant):  # noqa: F811
    usage, _ = compiled[("gemm_narrow_variant.hip", variant)]
    kernels = {k: u for k, u in usage.items() if "gemm_direct_kernel" in k}
    assert len(kernels) == 5, list(usage)  # two tiles of either precision, and one whose waves share the rows' operands
    for name, u in kernels.items():
        assert u["VGPRs"] <= 256 and u["AGPRs"] == 0 and u["ScratchSize"] == 0 and u["Occupancy"] >= 2, (name, u)


# On either side of the lines between the few-rows kernel and the large tiles that the factors in choose_direct draw.
@pytest.mark.parametrize("kind,M,K,N,fp4,few", [
    ("plain", 1131, 2048, 10112, True, 2), ("plain", 4608, 15360, 3072, True, 0), ("rope", 1614, 3968, 11904, True, 2), ("next", 2154, 1792, 7168, True, 2),
    ("plain", 225, 4992, 10624, False, 2), ("plain", 175, 9984, 14976, False, 2), ("plain", 261, 1152, 14208, False, 0), ("next", 1486, 1024, 4096, False, 0),
    ("next", 1486, 2048, 8192, False, 0),
])
def test_few_rows_or_large_tiles(kind, M, K, N, fp4, few):
    assert plan_of(call(kind, M, K, N, 32, fp4)).few_rows == few


# The lines that rank, epilogue and the rows' length draw between the NVFP4 few-rows kernel and whole large tiles, in one round and in several.
@pytest.mark.parametrize("kind,M,K,N,R,few", [
    ("plain", 10224, 1152, 3072, 160, 0), ("plain", 3771, 1152, 3072, 128, 0), ("plain", 1049, 1152, 13056, 160, 0), ("rope", 3662, 1024, 3456, 160, 0),
    ("silu", 20295, 1280, 12416, 128, 0), ("split", 1857, 896, 6912, 128, 0), ("plain", 1836, 12032, 5888, 32, 2), ("plain", 1131, 2048, 10112, 32, 2),
    ("split", 711, 10624, 14976, 32, 2), ("silu", 1129, 4224, 9472, 64, 2), ("next", 2154, 1792, 7168, 32, 2), ("silu", 1098, 1792, 12288, 48, 2),
    ("plain", 901, 4736, 11264, 128, 2), ("plain", 2972, 1792, 4864, 128, 0), ("plain", 8470, 1280, 3584, 128, 0), ("plain", 4608, 3072, 21504, 32, 0),
    ("plain", 4608, 15360, 3072, 32, 0), ("plain", 2666, 1664, 15360, 48, 2), ("rope", 3877, 2304, 14208, 16, 2), ("next", 4178, 2432, 16512, 16, 2),
    ("litela", 1280, 3072, 8448, 128, 2), ("split", 1280, 1152, 8448, 32, 2),
])
def test_nvfp4_few_rows_or_large_tiles_by_rank(kind, M, K, N, R, few):
    assert plan_of(call(kind, M, K, N, R, True)).few_rows == few


# (few_rows, shared_rows) on either side of the lines of the shared-rows form: the tiles per compute unit, and the other forms where these are faster.
@pytest.mark.parametrize("kind,M,K,N,R,want", [
    ("rope", 256, 3072, 9216, 32, (2, 1)), ("rope", 505, 2048, 6144, 128, (2, 1)), ("rope", 505, 3072, 9216, 32, (0, 0)), ("plain", 384, 3072, 9216, 32, (2, 1)),
    ("next", 256, 3072, 12288, 32, (2, 1)), ("next", 256, 3072, 12288, 128, (2, 1)), ("next", 505, 3072, 12288, 128, (0, 0)), ("next", 1280, 1152, 4608, 128, (0, 0)),
    ("next", 4357, 1024, 1152, 128, (0, 0)), ("silu", 408, 512, 4864, 96, (1, 0)), ("silu", 607, 2176, 3328, 0, (1, 0)), ("rope", 347, 4992, 5760, 32, (1, 0)),
    ("split", 196, 12416, 10752, 128, (2, 1)), ("next", 585, 11392, 4224, 64, (2, 1)), ("next", 1641, 8192, 2560, 32, (2, 1)), ("split", 1280, 128, 3072, 32, (2, 0)),
])
def test_where_waves_share_the_rows(kind, M, K, N, R, want):
    p = plan_of(call(kind, M, K, N, R, False))
    assert (p.few_rows, p.shared_rows) == want, p


@pytest.mark.parametrize("variant", [0, 1])
def test_waits_for_the_copies_of_shared_rows(compiled, variant):  # noqa: F811
    """The kernels whose waves share the rows' operands wait for an asynchronous copy by the number of requests made after it: three for
    the columns behind every copy, none dropped, none of another kind between them."""
    _, lines = compiled[("gemm_narrow_variant.hip", variant)]
    text = "\n".join(lines)
    start = next(m.start() for m in re.finditer(r"^_ZN\S*gemm_direct_kernelILb0ELi2ELi1ELi4E\S*:", text, re.M))
    body = text[start:text.index("s_endpgm", start)].split("\n")
    ops = []
    for line in body:
        t = line.strip()
        wait = re.match(r"s_waitcnt vmcnt\((\d+)\) lgkmcnt\(0\)$", t)
        if t.startswith("global_load_lds"):
            ops.append("C")
        elif re.match(r"(global|buffer|flat|scratch)_(load|store|atomic)", t):
            ops.append("w")
        elif wait and int(wait[1]) % 4 == 3:
            ops.append(str(int(wait[1]) // 4))
        elif t.startswith("s_barrier"):
            ops.append("B")
    main = "".join(ops)
    main = main[:main.index("0B") + 2]  # (the last wait leaves the last k-group's own requests)
    assert re.fullmatch(r"((Cwww)+2B|1B|0B)+", main), main
    assert set(re.findall(r"(?:Cwww)+", main)) <= {"Cwww", "Cwww" * 3}, main  # a k-group's, or the first three k-groups'
    assert re.search(r"2B1B0B$", main), main


def test_addresses_of_shared_rows():
    """The asynchronous copies of a k-group's rows (three KB of two fragments, 128 bytes of scales) and the columns' operands."""
    for M, K, N in ((1, 256, 128), (100, 640, 768), (505, 3072, 6144), (1153, 512, 3072)):
        M_pad, kgroups, padded = (M + 255) // 256 * 256, K // 64, (N + 255) // 256 * 256
        act_bytes, asc_bytes, wgt_bytes, wsc_bytes = M_pad * K * 3 // 4, kgroups * M_pad * 2, padded * K * 3 // 4, padded // 256 * kgroups * 2048
        for f0 in range(0, (M + 63) // 64 * 2, 2):
            for g in (0, kgroups - 1):
                first = (f0 // 4 * kgroups + g) * 4 * FRAG + f0 % 4 * FRAG
                assert first % 16 == 0 and first + 2 * 1024 + 63 * 16 + 16 == first + 2 * FRAG <= act_bytes
                assert (g * M_pad + f0 * 32) * 2 % 16 == 0 and (g * M_pad + f0 * 32) * 2 + 7 * 16 + 16 <= asc_bytes
        for nb in range(N // 128):
            for wave in range(4):
                tile = nb % 2 * 4 + wave
                assert (nb // 2 * kgroups + kgroups - 1) * 8 * FRAG + tile * FRAG + 1024 + 63 * 8 + 8 <= wgt_bytes
                assert (nb // 2 * kgroups + kgroups - 1) * 2048 + tile * 256 + 31 * 8 + 4 <= wsc_bytes


def test_nvfp4_large_tiles_that_few_rows_calls_could_take_need_no_workspace():
    """Where the models would have the large tiles, but so few of them that they are split along K, the few-rows kernel stays: a program may
    capture its call without a call before."""
    for kind, M, K, N in (("plain", 1214, 3456, 5760), ("plain", 1763, 5888, 3584), ("silu", 2263, 2816, 2944)):
        p = plan_of(call(kind, M, K, N, 512, True))
        assert p.few_rows == 2 and not p.shared_tiles, p
