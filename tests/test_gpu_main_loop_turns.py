"""The INT4 GEMM's main loop in whole turns of its LDS ring (three k-groups a turn, the rest behind them one by one) at every
remainder, whole and split along K (odd counts of k-groups), against the oracle; and launches with at most one 128-row tile per
compute unit and 64-row tiles next to them against whole tiles only: the same bits."""

import pytest
import torch

from conftest import announce
from gpu_util import check_output, make_module, make_oracle, record_plans
from oracle import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [128, 256, 384, 512, 640, 768, 896, 1024])
def test_every_remainder(dev, K, monkeypatch):
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"turns K={K}")
    layer = synth.make_layer(256, K, 16, seed=K)
    m, ref = make_module(layer, dev), make_oracle(layer)
    x = synth.make_activations(256, K, seed=K)
    act, asc, la = m.quantize(x.to(dev))
    want = ref.forward_quant(*ref.quantize(x))[:256]
    for parts in (1, 2, 3):  # K / 64 is even: 2 or 3 parts have odd counts of k-groups among them
        monkeypatch.setattr(gemm_mod, "K_SPLIT", parts)
        out = torch.full((256, 256), float("nan"), dtype=torch.bfloat16, device=dev)
        m.forward_quant(act, asc, la, out)
        torch.cuda.synchronize()
        check_output(out, want)


@pytest.mark.parametrize("kind,M,K,N", [("plain", 1024, 128, 9216), ("plain", 1000, 384, 9216), ("plain", 1024, 896, 9216), ("next", 1024, 640, 9216)])
def test_one_whole_tile_per_unit_and_half_ones(dev, kind, M, K, N, monkeypatch):
    from nunchaku_amd import packing
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"both heights {kind} M={M} K={K} N={N}")
    m, nxt = make_module(synth.make_layer(N, K, 32, seed=K), dev), make_module(synth.make_layer(128, N, 32, seed=9), dev)
    t, n = m.native_tensors(), nxt.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    plans = record_plans(monkeypatch, dev)

    def run(split):
        monkeypatch.setattr(gemm_mod, "K_SPLIT", split)
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
        outs = dict(out=out)
        if kind == "next":
            outs.update(qout=torch.zeros(act.shape[0], packing.act_nbytes_per_row(N, False), dtype=torch.uint8, device=dev),
                        oscales=torch.zeros(N // 64, act.shape[0], dtype=torch.bfloat16, device=dev), lora_act_out=torch.zeros(act.shape[0], 32, device=dev))
        extra = dict(lora_down=n["proj_down"], smooth_factor=n["smooth_factor"]) if kind == "next" else {}
        gemm_mod.svdq_gemm_w4a4(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=t["bias"], lora_act_in=la, lora_up=t["proj_up"], **outs, **extra)
        torch.cuda.synchronize()
        return {k: v.cpu() for k, v in outs.items()}

    want, got = run(1), run(None)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        p = plans[-1]
        assert p.few_rows == 0 and p.half_blocks > 0 and 0 < p.full_blocks * (N // 256) <= 256, p
    for name in got:
        assert torch.equal(got[name].view(torch.uint8), want[name].view(torch.uint8)), name
