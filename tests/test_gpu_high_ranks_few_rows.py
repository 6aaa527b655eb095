"""NVFP4 few-rows GEMM at ranks above 32 in tiles of 128 columns, whose low-rank operands come through LDS (csrc/gemm_direct_kernel.h, RANKS), against the large
tiles on the same operands: odd and even counts of 16-rank steps, the most that fit at once (8 beside 64 rows, 10 beside 32) and more, both heights, every epilogue."""

import pytest
import torch

from test_build_guard import compiled  # noqa: F401  (the fixture)
from test_gpu_few_rows import _compare

# (epilogue, M, K, N, R, 32-row blocks of a tile)
CASES = [
    ("silu", 33, 256, 256, 48, 1), ("next", 65, 384, 256, 160, 1), ("rope", 40, 640, 384, 176, 1), ("litela", 256, 256, 384, 80, 1), ("silu", 31, 128, 128, 272, 1),
    ("plain", 1300, 1152, 3072, 48, 2), ("plain", 929, 1024, 4608, 144, 2), ("next", 1186, 896, 2304, 128, 2), ("rope", 1263, 384, 2304, 112, 2), ("split", 1280, 384, 2304, 64, 2),
    ("silu", 1423, 640, 3072, 256, 2),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,K,N,R,mt", CASES)
def test_against_large_tiles(dev, kind, M, K, N, R, mt, monkeypatch):
    plan = _compare(dev, kind, M, K, N, R, True, monkeypatch)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert (plan.few_rows, plan.columns) == (mt, 128), plan


@pytest.mark.parametrize("variant", [0, 1])
def test_fits_its_registers(compiled, variant):  # noqa: F811
    usage, _ = compiled[("gemm_direct_ranks_variant.hip", variant)]
    kernels = {k: u for k, u in usage.items() if "gemm_direct_kernel" in k}
    assert len(kernels) == 2, list(usage)  # tiles of 32 and of 64 rows
    for name, u in kernels.items():
        assert u["VGPRs"] <= 256 and u["AGPRs"] == 0 and u["ScratchSize"] == 0 and u["Occupancy"] >= 2, (name, u)


def test_copies_stay_inside_their_buffers():
    """The asynchronous copies of a chunk of 32 ranks: 16 bytes a lane, lora_up [N][R] bf16 and lora_act [M_pad][R] fp32, into the place of the sums."""
    for R in range(48, 1025, 16):
        nsteps = R // 16
        for MT in (1, 2):
            chunk = 128 * 64 + MT * 32 * 128
            copied = min(nsteps, 2 * (4 * 4 * 4096 // chunk))
            assert (copied + 1) // 2 * chunk <= 4 * 4 * 4096
            seen_up, seen_act = set(), set()
            for c in range((copied + 1) // 2):
                half = nsteps - 2 * c < 2
                for lane in range(64):
                    for block in range(8):
                        col, piece = block * 16 + lane // 4, (lane & 3) ^ ((block * 16 + lane // 4) >> 2 & 3)
                        off = col * R * 2 + c * 64 + (piece & 1 if half else piece) * 16
                        assert off + 16 <= (col + 1) * R * 2
                        seen_up.add((c, col, piece))
                    for block in range(4 * MT):
                        row = block * 8 + lane // 8
                        piece = (lane & 7) ^ (row >> 1 & 7)
                        off = row * R * 4 + c * 128 + (piece & 3 if half else piece) * 16
                        assert off + 16 <= (row + 1) * R * 4
                        seen_act.add((c, row, piece))
            assert len(seen_up) == (copied + 1) // 2 * 512 and len(seen_act) == (copied + 1) // 2 * 256 * MT
