"""NVFP4 few-rows GEMM with 64-row tiles and 32-row tiles behind them (csrc/gemm.hip, ``few_rows_heights``) against the large tiles on the same operands:
every epilogue, both parities of the blocks of 32 rows, rows that end inside a block, two to nine k-groups on four waves (rings of two and three)."""

import pytest
import torch

from test_gpu_few_rows import _compare

pytestmark = pytest.mark.gpu

# (epilogue, M, K, N, R, blocks of 64 rows on 256 compute units, blocks of 32 rows behind them)
CASES = [
    ("plain", 929, 1024, 4608, 16, 14, 2), ("plain", 841, 768, 5376, 48, 12, 3), ("silu", 555, 768, 7680, 0, 8, 2), ("silu", 1423, 640, 3072, 32, 21, 3),
    ("next", 877, 128, 4608, 16, 14, 4), ("next", 1186, 896, 2304, 80, 14, 12), ("rope", 596, 768, 3840, 48, 8, 3), ("rope", 1263, 640, 2304, 0, 14, 12),
    ("split", 512, 640, 4992, 80, 6, 4), ("split", 1280, 384, 2304, 0, 14, 12), ("litela", 1024, 256, 4608, 32, 14, 4), ("litela", 768, 1152, 5760, 16, 11, 2),
]


@pytest.mark.parametrize("kind,M,K,N,R,full,half", CASES)
def test_against_large_tiles(dev, kind, M, K, N, R, full, half, monkeypatch):
    plan = _compare(dev, kind, M, K, N, R, True, monkeypatch)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        rows = (M + 255) // 256 * 256 if kind == "next" else M  # (all padded rows; the others of such kinds end with a block of 256: rows behind them are NaN in out_k)
        assert (plan.few_rows, plan.columns, plan.full_blocks, (rows + 31) // 32 - 2 * plan.full_blocks) == (2, 128, full, half), plan
