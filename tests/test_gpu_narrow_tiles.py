"""The few-rows GEMM with the plain epilogue in every tile it chooses among (csrc/gemm.hip, ``plain_tile``) against the kernels with
large tiles (``K_SPLIT = 1``): rows and columns that end inside a tile, fewer k-groups than waves and counts that the ring of requests
does not divide, ranks 0 to 80, outputs narrower than the padded layer, and no byte written outside the output."""

import pytest
import torch

from conftest import announce
from gpu_util import Guarded, bf16_ulp, make_module, record_plans
from oracle import synth

pytestmark = pytest.mark.gpu

# (tile, M, K, N, R); a pair of tiles: INT4's and NVFP4's
CASES = [
    ((32, 32), 1, 128, 128, 16), ((32, 32), 31, 640, 384, 0), ((32, 32), 33, 384, 256, 48), ((32, 32), 64, 1664, 1152, 80),
    ((32, 64), 32, 1152, 12288, 32), (((32, 64), (32, 32)), 17, 128, 12416, 16), (((32, 64), (64, 32)), 97, 640, 4096, 48), ((64, 32), 128, 3072, 3072, 32),
    (((64, 64), (32, 32)), 256, 1152, 3072, 32), ((64, 64), 225, 2176, 3200, 0), ((64, 64), 300, 2304, 3072, 64),
    ((32, 128), 89, 2432, 20480, 32), ((64, 128), 1157, 640, 3072, 48), (((64, 128), (32, 64)), 505, 384, 3072, 48), (((64, 128), (32, 64)), 1000, 512, 1536, 0),
]
SHARED_ROWS = [(1157, 640, 3072)]  # (M, K, N) of INT4 launches whose waves share the rows' operands; those of all others split K


@pytest.mark.parametrize("fp4", [False, True])
@pytest.mark.parametrize("tile,M,K,N,R", CASES)
def test_against_large_tiles(dev, tile, M, K, N, R, fp4, monkeypatch):
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"narrow tiles {tile} M={M} K={K} N={N} R={R} fp4={fp4}")
    g = torch.Generator().manual_seed(M + K + N)
    layer = synth.make_layer(N, K, R, seed=K + N, fp4=fp4)
    layer.wcscales = (0.5 + torch.rand(N, generator=g)).to(torch.bfloat16) if fp4 else None
    m = make_module(layer, dev)
    t = m.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    kw = dict(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=t["bias"], fp4=fp4, alpha=m.alpha if fp4 else 1.5, wcscales=t["wcscales"])
    if R:
        kw.update(lora_act_in=la, lora_up=t["proj_up"], lora_scales=[0.5 + 0.25 * i for i in range((R + 15) // 16)])
    plans, outs = record_plans(monkeypatch, dev), []
    for split in (1, None, None):
        monkeypatch.setattr(gemm_mod, "K_SPLIT", split)
        out = Guarded((M, N - 8), torch.bfloat16, dev)  # (the last column tile ends 8 columns early)
        gemm_mod.svdq_gemm_w4a4(**kw, out=out.t)
        torch.cuda.synchronize()
        out.check("out")
        outs.append(out.t.cpu())
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        want = tile[fp4] if isinstance(tile[0], tuple) else tile
        assert plans[0].few_rows == 0 and all((32 * p.few_rows, p.columns) == want for p in plans[1:]), plans
        assert all(bool(p.shared_rows) == (not fp4 and (M, K, N) in SHARED_ROWS) for p in plans[1:]), plans
    assert torch.equal(outs[1].view(torch.int16), outs[2].view(torch.int16)), "changed between two launches"
    a, b = outs[1].float(), outs[0].float()
    # sums of K products and R more in another order: 2^-24 (K + R) of the largest value at most; then one rounding that may go
    # the other way
    tol = (K + R) * 2.0**-24 * b.abs().max()
    assert not torch.isnan(a).any()
    assert ((a - b).abs() <= torch.maximum(bf16_ulp(torch.maximum(a.abs(), b.abs())), tol)).all(), (a - b).abs().max()
    assert (a != b).float().mean().item() < 2e-2
