"""INT4 launches of two and a half to three tiles of 64 x 128 per compute unit, whose waves share the rows' operands (csrc/gemm.hip, ``staged_rows``), against
the large tiles on the same operands: every epilogue, one and three k-groups before the whole turns of the ring, ranks up to the last that takes it."""

import pytest
import torch

from plan_util import call, plan_of
from test_gpu_few_rows import _compare

CASES = [
    ("plain", 1301, 640, 4224, 64), ("plain", 2500, 256, 2304, 0), ("silu", 1301, 384, 4224, 48), ("next", 1216, 256, 4224, 32), ("next", 2555, 640, 2176, 16),
    ("rope", 1251, 384, 4224, 64), ("split", 1280, 640, 4224, 16), ("litela", 1280, 256, 4224, 32),
]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,K,N,R", CASES)
def test_against_large_tiles(dev, kind, M, K, N, R, monkeypatch):
    plan = _compare(dev, kind, M, K, N, R, False, monkeypatch)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert (plan.few_rows, plan.columns, plan.shared_rows) == (2, 128, 1), plan


# On either side of its lines: 2.5 and 3 tiles per compute unit, rank 64, 1024 columns, a split along K.
@pytest.mark.parametrize("kind,M,K,N,R,shared", [
    ("rope", 640, 3072, 9216, 32, 1), ("rope", 704, 3072, 9216, 32, 0), ("rope", 505, 3072, 9216, 32, 0), ("silu", 1301, 384, 4224, 64, 1), ("silu", 1301, 384, 4224, 80, 0),
    ("silu", 5100, 512, 1024, 32, 1), ("silu", 5820, 512, 896, 32, 0), ("plain", 1301, 1152, 4224, 32, 1), ("plain", 1301, 128, 4224, 32, 0),
])
def test_which_launches(kind, M, K, N, R, shared):
    p = plan_of(call(kind, M, K, N, R, False))
    assert p.shared_rows == shared, p


# Less than 2048 columns that are whole blocks of 256: up to K = 1408.
@pytest.mark.parametrize("kind,M,K,N,R,shared", [
    ("plain", 4184, 1408, 1280, 32, 1), ("plain", 4184, 1536, 1280, 32, 0), ("plain", 4184, 5376, 1280, 16, 0), ("silu", 5451, 5504, 1024, 32, 0), ("rope", 3700, 2304, 1536, 32, 0),
    ("plain", 4864, 5376, 1152, 32, 1), ("plain", 3000, 1536, 1920, 32, 1), ("plain", 2700, 5376, 2048, 32, 1), ("rope", 640, 15360, 9216, 32, 1), ("next", 1700, 15360, 3072, 16, 1),
])
def test_which_columns(kind, M, K, N, R, shared):
    p = plan_of(call(kind, M, K, N, R, False))
    assert p.shared_rows == shared, p
