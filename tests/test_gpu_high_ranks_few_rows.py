"""NVFP4 few-rows GEMM at ranks above 32 in tiles of 128 columns, whose low-rank operands come through LDS (csrc/gemm_direct_kernel.h, RANKS), against the large
tiles on the same operands: odd and even counts of 16-rank steps, the most that fit at once (8 beside 64 rows, 10 beside 32) and more, both heights, every epilogue."""

import pytest
import torch

from conftest import announce
from gpu_util import Guarded, make_module, record_plans
from oracle import synth
from plan_util import call, plan_of
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


# Odd numbers of 16-rank steps come wave by wave but for several tiles of 64 rows per compute unit (280 and 360 of them; 228 and 216 where there is one), rank 48 always.
@pytest.mark.parametrize("kind,M,K,N,R,mt,copied", [
    ("silu", 66, 640, 2688, 48, 1, 0), ("silu", 66, 640, 2688, 64, 1, 1), ("rope", 101, 640, 1536, 112, 1, 0), ("rope", 101, 640, 1536, 128, 1, 1), ("litela", 256, 640, 1152, 176, 1, 0),
    ("silu", 1216, 896, 1536, 80, 2, 0), ("silu", 1216, 896, 1536, 96, 2, 1), ("silu", 1263, 896, 1792, 80, 2, 1), ("silu", 1263, 896, 1792, 48, 2, 0), ("silu", 1263, 896, 2304, 144, 2, 1),
    ("rope", 760, 896, 2304, 144, 2, 0), ("silu", 1263, 896, 1792, 32, 2, 0),
])
def test_which_way(kind, M, K, N, R, mt, copied):
    p = plan_of(call(kind, M, K, N, R, True))
    assert (p.few_rows, p.columns, p.copied_ranks) == (mt, 128, copied), p
    assert plan_of(call(kind, M, K, N, R, False)).copied_ranks == 0


# Wave by wave or through LDS, both heights and two heights: the same products in the same order.  A step of zeros behind an odd number of them changes the way and no bit.
@pytest.mark.gpu
@pytest.mark.parametrize("silu,M,K,N,R", [(True, 40, 384, 256, 48), (True, 65, 640, 384, 80), (True, 31, 128, 128, 112), (True, 97, 256, 256, 176), (True, 1216, 896, 1536, 80),
                                          (True, 1263, 640, 1792, 48), (False, 1300, 1152, 3072, 48)])
def test_same_bits_either_way(dev, silu, M, K, N, R, monkeypatch):
    from nunchaku_amd import packing
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"ranks either way M={M} K={K} N={N} R={R}")
    m = make_module(synth.make_layer(N, K, R + 16, seed=K + N + R, fp4=True), dev)
    t = m.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    la[:, R:] = 0.0
    up = t["proj_up"]
    short = packing._tag(up[:, :R].contiguous(), "lora_up")
    plans, outs = record_plans(monkeypatch, dev), []
    for lora_act, lora_up in ((la, up), (la[:, :R].contiguous(), short)):
        out = Guarded((M, N), torch.bfloat16, dev)
        gemm_mod.svdq_gemm_w4a4(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=t["bias"], fp4=True, alpha=m.alpha, wcscales=t["wcscales"], lora_act_in=lora_act,
                                lora_up=lora_up, lora_scales=[0.5 + 0.125 * i for i in range(R // 16 + 1)], out=out.t, fuse_silu=silu)
        torch.cuda.synchronize()
        out.check("out")
        outs.append(out.t.float().cpu())
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert [p.copied_ranks for p in plans] == [1, 0] and plans[0].few_rows == plans[1].few_rows and plans[0].full_blocks == plans[1].full_blocks, plans
    assert not torch.isnan(outs[0]).any() and torch.equal(outs[0], outs[1])


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
