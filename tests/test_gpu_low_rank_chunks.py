"""The low-rank up projection of the GEMMs with large tiles takes its operands 32 ranks at a time through two buffers in LDS: ranks
that end in the middle of a chunk, at one, two, three and more chunks, the last column tile with half its columns, blocks of
64 rows, and the next layer's projection, whose operands take the buffers' place afterwards.  Against the oracle."""

import pytest
import torch

from conftest import announce
from gpu_util import check_output, make_module, make_oracle, off_alignment, record_plans
from oracle import linear as olin
from oracle import quant, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp4", [False, True])
@pytest.mark.parametrize("M,K,N,R,half_blocks", [(1, 128, 128, 16, 0), (300, 256, 384, 32, 0), (300, 128, 256, 48, 0), (256, 256, 128, 64, 0), (300, 128, 640, 80, 0),
                                                 (257, 128, 384, 144, 0), (257, 128, 384, 256, 0), (640, 128, 6144, 48, 1), (640, 128, 6144, 80, 1)])
def test_up_projection(dev, M, K, N, R, half_blocks, fp4, monkeypatch):
    from nunchaku_amd import packing
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"low-rank chunks M={M} K={K} N={N} R={R} fp4={fp4}")
    layer = synth.make_layer(N, K, R, seed=M + N + R, fp4=fp4)
    layer.wcscales = (0.5 + torch.rand(N, generator=torch.Generator().manual_seed(R))).to(torch.bfloat16) if fp4 else None
    m, ref = make_module(layer, dev), make_oracle(layer)
    t = m.native_tensors()
    x = synth.make_activations(M, K, seed=M)
    act, asc, _ = m.quantize(x.to(dev))
    M_pad = act.shape[0]
    lora_act = 3 * torch.randn(M_pad, R, generator=torch.Generator().manual_seed(N))
    lora_scales = [0.5 + 0.25 * i for i in range(R // 16)]
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    monkeypatch.setattr(gemm_mod, "K_SPLIT", None if half_blocks else 1)
    plans = record_plans(monkeypatch, dev)
    kw = dict(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=off_alignment(t["bias"]), fp4=fp4, alpha=m.alpha if fp4 else 1.5, wcscales=t["wcscales"],
              lora_act_in=lora_act.to(dev), lora_up=t["proj_up"], lora_scales=lora_scales)
    gemm_mod.svdq_gemm_w4a4(**kw, out=out)
    torch.cuda.synchronize()
    assert plans[-1].few_rows == 0
    if half_blocks and not fp4 and torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert plans[-1].half_blocks > 0
    codes, scales, _ = ref.quantize(x)
    a = quant.dequant_nvfp4(codes, scales) if fp4 else quant.dequant_int4(codes, scales)
    want = olin.gemm_w4a4(a, ref.w_deq, bias=layer.bias, lora_act_in=lora_act, lora_up=layer.proj_up, lora_scales=lora_scales, alpha=m.alpha if fp4 else 1.5,
                          wcscales=layer.wcscales)[:M]
    check_output(out, want)
    # the same product with the next layer's projection (rank 32: its operands wait in LDS; 48: they do not)
    for R_down in (32, 48):
        nxt = make_module(synth.make_layer(128, N, R_down, seed=9, fp4=fp4), dev).native_tensors()
        M_all = torch.empty(M_pad, N, dtype=torch.bfloat16, device=dev)
        down = torch.full((M_pad, R_down), float("nan"), dtype=torch.float32, device=dev)
        G = 16 if fp4 else 64
        gemm_mod.svdq_gemm_w4a4(**kw, out=M_all, qout=torch.empty(M_pad, packing.act_nbytes_per_row(N, fp4), dtype=torch.uint8, device=dev),
                                oscales=torch.empty(N // G, M_pad, dtype=torch.float8_e4m3fn if fp4 else torch.bfloat16, device=dev), lora_act_out=down,
                                lora_down=nxt["proj_down"], smooth_factor=nxt["smooth_factor"])
        torch.cuda.synchronize()
        check_output(M_all[:M], torch.nn.functional.gelu(want, approximate="tanh"))
        # the projection of the bf16 tile stored next to it: N products summed in fp32 in another order
        proj = synth.make_layer(128, N, R_down, seed=9, fp4=fp4).proj_down.double()
        wanted = M_all.cpu().double() @ proj
        bound = N * 2.0**-24 * (M_all.cpu().double().abs() @ proj.abs())
        assert ((down.cpu().double() - wanted).abs() <= bound).all()
