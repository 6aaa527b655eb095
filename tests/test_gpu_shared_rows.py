"""The INT4 few-rows GEMM whose waves share the rows' operands through LDS (csrc/gemm_direct_kernel.h, ``staged_rows`` in csrc/gemm.hip):
both remainders that an even number of k-groups leaves by its ring of four (one and three, before the whole turns), the fewest it
takes, rows that end inside a tile; the same bits as one wave per tile adds up (the large tiles: the same order of the k-groups) where the
epilogue is plain.  (The other epilogues: test_gpu_few_rows.py.)"""

import pytest
import torch

from conftest import announce
from gpu_util import Guarded, make_module, record_plans
from oracle import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [256, 384, 512, 640, 768, 896, 1152])
@pytest.mark.parametrize("M,N", [(1089, 3072), (1280, 3200)])  # 432 and 500 tiles of 64 x 128
def test_against_large_tiles(dev, M, N, K, monkeypatch):
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"shared rows M={M} K={K} N={N}")
    m = make_module(synth.make_layer(N, K, 48, seed=K + N), dev)
    t = m.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    kw = dict(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=t["bias"], lora_act_in=la, lora_up=t["proj_up"], lora_scales=[0.5, 0.75, 1.0])
    plans, outs = record_plans(monkeypatch, dev), []
    for split in (1, None, None):
        monkeypatch.setattr(gemm_mod, "K_SPLIT", split)
        out = Guarded((M, N), torch.bfloat16, dev)
        gemm_mod.svdq_gemm_w4a4(**kw, out=out.t)
        torch.cuda.synchronize()
        out.check("out")
        outs.append(out.t.cpu())
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert plans[0].few_rows == 0 and plans[1].few_rows == 2 and plans[1].shared_rows, plans
    assert torch.equal(outs[1].view(torch.int16), outs[2].view(torch.int16))
    # the main sums have the same bits; bias and low-rank term are added in one order too, the low-rank products 16 ranks at a time
    a, b = outs[1].float(), outs[0].float()
    assert not torch.isnan(a).any() and (a - b).norm() <= 2.0**-9 * 1e-2 * b.norm() and (a != b).float().mean().item() < 1e-3


# What the epilogue needs of its own is copied to LDS beside the stages: ranks that end inside a chunk of 32 and beyond the three chunks that are copied, with and without
# bias and per-column scales, and the epilogues of the other kernel.
@pytest.mark.parametrize("R,bias,scales,silu", [(16, True, True, False), (32, False, True, True), (48, True, False, True), (64, False, False, False), (96, True, True, True),
                                                (112, True, True, False), (160, True, True, True)])
def test_operands_of_the_epilogue(dev, R, bias, scales, silu, monkeypatch):
    from nunchaku_amd.ops import gemm as gemm_mod

    M, K, N = 1089, 640, 3072
    announce(f"shared rows, epilogue R={R} bias={bias} scales={scales} silu={silu}")
    m = make_module(synth.make_layer(N, K, R, seed=R), dev)
    t = m.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    wc = (0.5 + torch.rand(N, generator=torch.Generator().manual_seed(R))).to(torch.bfloat16).to(dev) if scales else None
    kw = dict(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=t["bias"] if bias else None, wcscales=wc, alpha=1.25, lora_act_in=la, lora_up=t["proj_up"],
              lora_scales=[0.5 + 0.125 * i for i in range(R // 16)], fuse_silu=silu)
    plans, outs = record_plans(monkeypatch, dev), []
    for split in (1, None, None):
        monkeypatch.setattr(gemm_mod, "K_SPLIT", split)
        out = Guarded((M, N), torch.bfloat16, dev)
        gemm_mod.svdq_gemm_w4a4(**kw, out=out.t)
        torch.cuda.synchronize()
        out.check("out")
        outs.append(out.t.cpu())
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert plans[0].few_rows == 0 and plans[1].few_rows == 2 and plans[1].shared_rows, plans
    assert torch.equal(outs[1].view(torch.int16), outs[2].view(torch.int16))
    # (the same sums in the same order, bias and activation after them: what differs is a rounding to bf16 that goes the other way, of few values)
    a, b = outs[1].float(), outs[0].float()
    assert not torch.isnan(a).any() and (a - b).norm() <= 2.0**-9 * 1e-2 * b.norm() and (a != b).float().mean().item() < 1e-3
