"""NVFP4 few-rows GEMM with 64-row tiles and 32-row tiles behind them (csrc/gemm.hip, ``few_rows_heights``) against the large tiles on the same operands:
every epilogue, both parities of the blocks of 32 rows, rows that end inside a block, two to nine k-groups on four waves (rings of two and three)."""

import pytest
import torch

from conftest import announce
from gpu_util import make_module, record_plans
from oracle import synth
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


# The rows of a launch of two heights, 256 at a time in launches of one: the same products in the same order, so the same bits.  (Codes and scales stand 32 rows at a time, [K/64][rows][4].)
@pytest.mark.parametrize("kind,M,K,N,R", [("plain", 929, 1024, 4608, 16), ("silu", 1423, 640, 3072, 32), ("next", 1186, 896, 2304, 80), ("rope", 596, 768, 3840, 48), ("silu", 1490, 896, 1792, 128)])
def test_same_bits_as_one_height(dev, kind, M, K, N, R, monkeypatch):
    from nunchaku_amd import packing
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"two heights, same bits {kind} M={M} K={K} N={N} R={R}")
    g = torch.Generator().manual_seed(M)
    m = make_module(synth.make_layer(N, K, R, seed=K + N, fp4=True), dev)
    t = m.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    M_pad = act.shape[0]
    ang = 6.283 * torch.rand(M_pad, 64, generator=g)
    table = torch.stack((ang.sin(), ang.cos()), dim=-1).reshape(M_pad, 128).to(dev)
    norm = (1.0 + 0.2 * torch.randn(128, generator=g)).to(torch.bfloat16).to(dev)
    smooth = make_module(synth.make_layer(128, N, 16, seed=9, fp4=True), dev).native_tensors()["smooth_factor"]

    def scales(s, a, b):  # of rows a ... b
        return s.view(torch.uint8).view(-1, M_pad, 4)[:, a:b].contiguous()

    def run(a, b):
        rows, pad = min(b, M) - a, b - a
        out = torch.full((pad if kind == "next" else rows, N), float("nan"), dtype=torch.bfloat16, device=dev)
        kw = {}
        if kind == "rope":
            kw = dict(norm_q=norm, norm_k=norm, rotary_emb=packing.repack_rotemb(table[a:b].contiguous()))
        if kind == "next":
            kw = dict(qout=torch.empty(pad, N // 2, dtype=torch.uint8, device=dev), oscales=torch.empty(N // 16, pad, dtype=torch.float8_e4m3fn, device=dev), smooth_factor=smooth)
        gemm_mod.svdq_gemm_w4a4(act=act[a:b], wgt=t["qweight"], ascales=scales(asc, a, b).view(torch.float8_e4m3fn).view(K // 16, pad), wscales=t["wscales"], bias=t["bias"], fp4=True,
                                alpha=m.alpha, wcscales=t["wcscales"], lora_act_in=la[a:b], lora_up=t["proj_up"], lora_scales=[0.5 + 0.125 * i for i in range(R // 16)], out=out,
                                fuse_silu=kind == "silu", **kw)
        torch.cuda.synchronize()
        return out, kw.get("qout"), kw.get("oscales")

    plans = record_plans(monkeypatch, dev)
    whole, parts = run(0, M_pad), [(a, run(a, a + 256)) for a in range(0, M_pad, 256)]
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert plans[0].low_blocks > 0 and all(p.few_rows and not p.low_blocks for p in plans[1:]), plans
    for a, (out, qout, oscales) in parts:
        assert not torch.isnan(out).any() and torch.equal(out.view(torch.int16), whole[0][a:a + 256].view(torch.int16)), a
        if kind == "next":
            assert torch.equal(qout, whole[1][a:a + 256]) and torch.equal(oscales.view(torch.uint8).view(-1, 256, 4), scales(whole[2], a, a + 256)), a
