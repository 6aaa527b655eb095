"""How the library divides a GEMM launch (csrc/gemm.hip, make_plan; csrc/gemm_params.h, tile_of), asked of the library itself:
every tile of an INT4 launch is taken by exactly one workgroup, whatever the numbers of 128-row and 64-row blocks; the rows a
launch divides into blocks are covered without leaving the padded tensor; each kernel is still chosen where its tests and its
measurements place it, and the same one with an allocated workspace and with the fixed one."""

import pytest

from plan_util import Plan, call, plan_of, tile_of


@pytest.mark.parametrize("nblocks", [1, 3, 12, 27, 36, 48])
def test_every_tile_once(nblocks):
    for full in (0, 1, 2, 7, 9, 10, 11, 36):
        for half in (0, 1, 2, 5, 20, 21):
            for kparts in ((1, 3) if half == 0 else (1,)):
                plan = Plan(full_blocks=full, half_blocks=half, kparts=kparts)
                total = (full * kparts + half) * nblocks
                tiles = [tile_of(plan, 256 * nblocks, b) for b in range(total)]
                got = [(t.row, t.column_block, t.part, t.rows) for t in tiles]
                want = {(mb * 128, nb, part, 128) for mb in range(full) for nb in range(nblocks) for part in range(kparts)}
                want |= {(full * 128 + mb * 64, nb, 0, 64) for mb in range(half) for nb in range(nblocks)}
                assert len(set(got)) == total and set(got) == want, (full, half, kparts)
                # the slots of the workspace: one number per tile for its parts to meet under, one per row block for its sums
                assert all(0 <= t.tile < full * nblocks for t in tiles if t.rows == 128)
                assert len({t.tile for t in tiles if t.rows == 128}) == full * nblocks
                assert all(t.row_block == (t.row // 128 if t.rows == 128 else full + (t.row - full * 128) // 64) for t in tiles)


@pytest.mark.parametrize("kind,K", [("plain", 128), ("plain", 3072), ("plain", 12288), ("rope", 3072)])
def test_rows_are_covered_inside_the_padded_tensor(kind, K):
    for fp4 in (False, True):
        for nblocks in (3, 12, 27, 36, 48, 84):
            for rows in [*range(1, 2200, 37), 4096, 4608, 9216, 18432, 18433]:
                p = plan_of(call(kind, rows, K, 256 * nblocks, 32, fp4))
                m_pad = (rows + 255) // 256 * 256
                if p.few_rows:
                    covered, height = p.row_blocks * 32 * p.few_rows, 32 * p.few_rows
                elif fp4:
                    assert 0 < p.workgroups <= 256 and p.shared_tiles == (m_pad // 256 * nblocks % p.workgroups != 0)
                    continue
                else:
                    covered, height = p.full_blocks * 128 + p.half_blocks * 64, 128
                    if p.kparts > 1:  # (whole tiles of all padded rows)
                        assert covered == m_pad and p.half_blocks == 0
                        continue
                assert rows <= covered <= m_pad and covered - rows < height


def test_rows_of_a_call_without_out():
    """The rows that svdq_gemm_w4a4_rows names limit what is worked out; without it, and with more than one output, all are."""
    for kind, with_out, rows, want in (("next", False, 300, 10), ("next", False, 0, 16), ("next", True, 0, 16), ("litela", True, 0, 16), ("split", True, 0, 16), ("plain", True, 0, 10)):
        p = plan_of(call(kind, 300, 256, 768, 32, False, with_out=with_out), rows=rows)
        assert (p.few_rows, p.row_blocks) == (1, want), (kind, p)


# Where the kernels meet on 256 compute units: sizes on either side of the lines that the comments at choose_direct,
# choose_row_blocks, choose_kparts and whole_tiles_fp4 give measurements for.
@pytest.mark.parametrize("kind,M,K,N,fp4,want", [
    ("plain", 256, 3072, 3072, False, dict(few_rows=2, columns=64)), ("plain", 1157, 3072, 3072, False, dict(few_rows=2, columns=128, shared_rows=1)), ("plain", 505, 3072, 9216, False, dict(half_blocks=8)),
    ("plain", 256, 12288, 3072, False, dict(few_rows=2, columns=64)), ("plain", 505, 12288, 3072, False, dict(few_rows=2, columns=128)), ("plain", 1536, 6144, 1536, False, dict(kparts=3)),
    ("plain", 4608, 3072, 9216, False, dict(full_blocks=35, half_blocks=2)), ("plain", 4608, 3072, 12288, False, dict(full_blocks=36)),
    # (slower in blocks of two heights than in whole tiles: they would fit exactly by an even finish that the hardware does not reach)
    ("plain", 4096, 3072, 9216, False, dict(full_blocks=32)), ("rope", 4096, 6144, 9216, False, dict(full_blocks=32)), ("plain", 2048, 3072, 18432, False, dict(full_blocks=16)),
    ("plain", 300, 3072, 3072, True, dict(few_rows=2, columns=64)), ("plain", 1157, 12288, 3072, True, dict(few_rows=2)), ("plain", 4608, 3072, 21504, True, dict(workgroups=252)),
    ("plain", 4608, 15360, 3072, True, dict(workgroups=216)), ("plain", 4608, 3072, 4608, True, dict(workgroups=256, shared_tiles=1)),
    # (short rows: whole large tiles, but not shared ones, whose workspace the fixed scratch has not)
    ("plain", 4608, 384, 9088, True, dict(workgroups=216)), ("plain", 6400, 640, 16384, True, dict(few_rows=2)),
    ("plain", 11008, 1024, 8576, True, dict(few_rows=2)), ("rope", 4096, 384, 14592, True, dict(workgroups=228)), ("next", 4096, 3072, 6144, True, dict(few_rows=2)),
    ("next", 2304, 256, 7680, True, dict(few_rows=2)), ("next", 4608, 4096, 4608, True, dict(workgroups=256, shared_tiles=1)),
])
def test_which_kernel(kind, M, K, N, fp4, want):
    p = plan_of(call(kind, M, K, N, 32, fp4))
    for name in ("few_rows", "half_blocks", "kparts", "shared_tiles", *want):
        default = 1 if name == "kparts" and not fp4 and not p.few_rows else 0
        assert getattr(p, name) == want.get(name, default), p


def test_operands_off_their_alignment_take_the_large_tiles():
    """The few-rows kernel reads bias, wcscales and the output scales 8 bytes at a time and colnorm 16."""
    for fp4 in (False, True):
        assert plan_of(call("next", 256, 3072, 3072, 32, fp4)).few_rows
        for field, off in (("bias", 2), ("bias", 4), ("wcscales", 2), ("oscales", 4), ("colnorm", 8)):
            a = call("next", 256, 3072, 3072, 32, fp4)
            setattr(a, field, (1 << 20) + off)
            assert not plan_of(a).few_rows, field
    # NVFP4 then splits few tiles among parties of equal size
    assert plan_of(call("plain", 256, 3072, 3072, 32, True, aligned=False)).workgroups == 24
    assert plan_of(call("plain", 256, 12288, 3072, 32, True, aligned=False)).workgroups == 48


def test_k_split_asks_for_large_tiles():
    assert plan_of(call("plain", 256, 3072, 3072, 32, False, k_split=1)).kparts == 1
    assert plan_of(call("plain", 256, 3072, 3072, 32, False, k_split=6)).kparts == 6
    assert plan_of(call("plain", 256, 128, 3072, 32, False, k_split=6)).kparts == 2  # (one k-group each at least)
    assert plan_of(call("plain", 256, 3072, 3072, 32, True, k_split=1)).workgroups == 12
    assert plan_of(call("plain", 256, 3072, 3072, 32, True, k_split=3)).workgroups == 36


def test_shares_that_only_larger_tiles_fit_into_the_fixed_scratch():
    assert plan_of(call("next", 256, 128, 12288, 16, False, R_down=832)).few_rows  # 96 shares of 128 columns: 81.8 MB
    assert not plan_of(call("next", 256, 128, 12288, 16, False, R_down=1024)).few_rows  # 100.7 MB; 48 of 256 columns: 50.3
    assert plan_of(call("next", 512, 128, 12288, 16, False, R_down=1024, with_out=False), rows=1).few_rows  # 201 and 101 MB: neither fits
    assert plan_of(call("next", 256, 128, 12288, 16, True, R_down=1024)).few_rows  # (NVFP4: as many in either kernel)
