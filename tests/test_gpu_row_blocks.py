"""INT4 GEMM with the last rows in tiles of 64 rows (csrc/gemm6_kernel.h, output_tile<.., 1>) against the same launch in tiles
of 128 rows (``K_SPLIT = 1``).  Every element is the same sum in the same order, so the outputs are the same bits; only the
linear-attention sums are added up in other pieces."""

import pytest
import torch

from conftest import announce
from gpu_util import make_module, record_plans
from oracle import synth

pytestmark = pytest.mark.gpu

# (epilogue, M, K, N, R): two k-groups (fewer than LDS stages) and more, both parities of the count of 64-row blocks, a ragged last
# column block, rows that end inside a 64-row block, 64-row tiles only, ranks on either side of the LDS-staged projection
CASES = [
    ("plain", 2049, 128, 8960, 16), ("plain", 2100, 256, 9216, 48), ("plain", 1536, 384, 12672, 0), ("plain", 4352, 640, 2688, 32), ("silu", 2304, 256, 8448, 32),
    ("next", 2049, 256, 8576, 32), ("next", 2304, 128, 8448, 48), ("rope", 2049, 256, 8832, 32), ("split", 2304, 128, 8448, 16), ("litela", 4096, 256, 6912, 32), ("litela", 2304, 384, 8448, 16),
]


@pytest.mark.parametrize("kind,M,K,N,R", CASES)
def test_same_bits_as_whole_tiles(dev, kind, M, K, N, R, monkeypatch):
    from nunchaku_amd import packing
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"row blocks {kind} M={M} K={K} N={N} R={R}")
    M_pad = (M + 255) // 256 * 256
    plans = record_plans(monkeypatch, dev)
    g = torch.Generator().manual_seed(M + K + N)
    layer = synth.make_layer(N, K, R, seed=K + N)
    m = make_module(layer, dev)
    t = m.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    kw = dict(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=t["bias"], alpha=1.5)
    if R:
        kw.update(lora_act_in=la, lora_up=t["proj_up"])
    new = lambda *shape, dtype=torch.bfloat16: torch.full(shape, float("nan"), dtype=dtype, device=dev)  # noqa: E731

    def run(split):
        monkeypatch.setattr(gemm_mod, "K_SPLIT", split)
        if kind in ("plain", "silu"):
            outs = dict(out=new(M, N))
            gemm_mod.svdq_gemm_w4a4(**kw, **outs, fuse_silu=kind == "silu")
        elif kind == "next":
            outs = dict(out=new(M_pad, N), qout=torch.zeros(M_pad, packing.act_nbytes_per_row(N, False), dtype=torch.uint8, device=dev),
                        oscales=new(N // 64, M_pad), lora_act_out=new(M_pad, R, dtype=torch.float32))
            gemm_mod.svdq_gemm_w4a4(**kw, **outs, lora_down=nxt["proj_down"], smooth_factor=nxt["smooth_factor"])
        elif kind in ("rope", "split"):
            outs = dict(out=new(M, N)) if kind == "rope" else {k: new(1, N // 384, M_pad, 128, dtype=torch.float16) for k in ("out_q", "out_k", "out_v")}
            gemm_mod.svdq_gemm_w4a4(**kw, **outs, norm_q=nq, norm_k=nq, rotary_emb=rot, attn_tokens=M if kind == "split" else 0)
        else:
            rows = 2048 if M_pad % 2048 == 0 else 256
            outs = dict(out_linearattn=new(M_pad // rows, rows, N // 3), out_vk=new(M_pad // rows, N // 96, 33, 32, dtype=torch.float32))
            gemm_mod.svdq_gemm_w4a4(**kw, **outs)
        torch.cuda.synchronize()
        return {k: v.cpu() for k, v in outs.items()}

    if kind == "next":
        nxt = make_module(synth.make_layer(128, N, R, seed=9), dev).native_tensors()
    if kind in ("rope", "split"):
        ang = 6.283 * torch.rand(M_pad, 64, generator=g)
        rot = packing.repack_rotemb(torch.stack((ang.sin(), ang.cos()), dim=-1).reshape(M_pad, 128).to(dev))
        nq = (1.0 + 0.2 * torch.randn(128, generator=g)).to(torch.bfloat16).to(dev)
    want, got = run(1), run(None)
    assert plans[0].half_blocks == 0 and plans[0].kparts == 1
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert plans[1].few_rows == 0 and plans[1].half_blocks > 0, "the case has no 64-row tiles"
    for name in got:
        a, b = got[name], want[name]
        if name == "out_vk":  # 256 or 2048 products per sum, added in other pieces: 2^-24 of the largest per addition
            rows = M_pad // a.shape[0]
            assert not torch.isnan(a).any()
            assert (a - b).abs().max() <= rows * 2.0**-24 * b.abs().max()
        else:
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), name
