"""The few-rows GEMM (csrc/gemm_direct_kernel.h) against the kernels with large tiles (``K_SPLIT = 1`` selects them) on the
same operands, at the sizes where its tiles end: one row, a row more or less than a block of 32 or 64, fewer k-groups than
waves and counts that its ring does not divide, one column tile and several, every epilogue, ranks up to 80."""

import pytest
import torch

from conftest import announce
from gpu_util import bf16_ulp, make_module, record_plans
from oracle import synth

pytestmark = pytest.mark.gpu

# (epilogue, M, K, N, R); the launcher takes 32-row tiles for the first two rows of this list, and 64-row tiles, on 256 compute
# units, for the others (plain epilogue: the tile that its model says, see test_gpu_narrow_tiles.py)
CASES = [
    ("plain", 1, 128, 128, 16), ("plain", 31, 128, 256, 0), ("plain", 33, 640, 384, 48), ("plain", 64, 1152, 128, 80), ("plain", 65, 256, 640, 32),
    ("silu", 96, 384, 256, 16), ("next", 33, 128, 128, 16), ("next", 97, 640, 384, 48), ("rope", 40, 384, 384, 32), ("split", 256, 256, 768, 16),
    ("litela", 256, 256, 384, 16),
    ("plain", 1200, 384, 3072, 32), ("next", 1185, 256, 3072, 32), ("rope", 1217, 256, 3072, 16), ("split", 1280, 128, 3072, 32), ("litela", 1024, 256, 3456, 32),
    ("plain", 1217, 640, 3072, 32), ("next", 1200, 1152, 3072, 48), ("rope", 1153, 512, 3072, 0),  # (NVFP4: 3 and 2, 5 and 4, 2 k-groups per wave)
]

# INT4, 64 x 128 tiles, on 256 compute units.  Two waves split K and two the columns: two to nine k-groups per wave, which its ring of two divides and does not.
SPLIT_K_CASES = [
    ("plain", 505, 384, 3072, 48), ("plain", 1000, 512, 1536, 16), ("plain", 1281, 640, 1152, 80), ("plain", 1500, 1152, 768, 32),
    ("next", 320, 256, 2304, 48), ("next", 769, 384, 1152, 16), ("next", 320, 640, 2304, 32), ("next", 769, 1152, 1152, 80), ("silu", 193, 384, 5376, 32),
    ("rope", 193, 640, 5376, 32), ("rope", 1000, 256, 1152, 0), ("split", 512, 384, 2304, 16), ("litela", 512, 512, 2304, 32), ("litela", 1024, 640, 1152, 32),
]
# The waves split the columns and share the rows: one and three k-groups before the whole turns of its ring, every epilogue but the plain one.
SHARED_ROWS_CASES = [
    ("next", 1185, 256, 3072, 32), ("next", 1200, 1152, 3072, 48), ("next", 1200, 384, 3072, 16), ("rope", 1217, 256, 3072, 16), ("rope", 1153, 640, 3072, 0),
    ("split", 1280, 256, 3072, 32), ("split", 1280, 384, 3072, 16), ("silu", 1200, 384, 3072, 0), ("silu", 1153, 512, 3072, 32), ("litela", 1024, 256, 3456, 32),
    ("litela", 1024, 384, 3456, 48),
]


@pytest.mark.parametrize("fp4", [False, True])
@pytest.mark.parametrize("kind,M,K,N,R", CASES)
def test_against_large_tiles(dev, kind, M, K, N, R, fp4, monkeypatch):
    plan = _compare(dev, kind, M, K, N, R, fp4, monkeypatch)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert plan.few_rows in ((1, 2) if kind == "plain" else (1,) if M <= 256 else (2,)), plan


@pytest.mark.parametrize("shared,case", [(0, c) for c in SPLIT_K_CASES] + [(1, c) for c in SHARED_ROWS_CASES])
def test_int4_64_x_128_tiles(dev, case, shared, monkeypatch):
    plan = _compare(dev, *case, False, monkeypatch)
    if torch.cuda.get_device_properties(dev).multi_processor_count == 256:
        assert (plan.few_rows, plan.columns, plan.shared_rows) == (2, 128, shared), plan


def _compare(dev, kind, M, K, N, R, fp4, monkeypatch):
    """Compares the launch that the library chooses with the large tiles' and returns its plan."""
    from nunchaku_amd import packing
    from nunchaku_amd.ops import gemm as gemm_mod

    announce(f"few rows {kind} M={M} K={K} N={N} R={R} fp4={fp4}")
    g = torch.Generator().manual_seed(M + K + N)
    layer = synth.make_layer(N, K, R, seed=K + N, fp4=fp4)
    layer.wcscales = (0.5 + torch.rand(N, generator=g)).to(torch.bfloat16) if fp4 else None
    m = make_module(layer, dev)
    t = m.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))
    M_pad = act.shape[0]
    kw = dict(act=act, wgt=t["qweight"], ascales=asc, wscales=t["wscales"], bias=t["bias"], fp4=fp4, alpha=m.alpha if fp4 else 1.5, wcscales=t["wcscales"])
    if R:
        kw.update(lora_act_in=la, lora_up=t["proj_up"], lora_scales=[0.5 + 0.25 * i for i in range((R + 15) // 16)])
    new = lambda *shape, dtype=torch.bfloat16: torch.full(shape, float("nan"), dtype=dtype, device=dev)  # noqa: E731
    plans = record_plans(monkeypatch, dev)

    def run(split):
        monkeypatch.setattr(gemm_mod, "K_SPLIT", split)
        if kind in ("plain", "silu"):
            outs = dict(out=new(M, N))
            gemm_mod.svdq_gemm_w4a4(**kw, **outs, fuse_silu=kind == "silu")
        elif kind == "next":
            G = 16 if fp4 else 64
            outs = dict(out=new(M_pad, N), qout=torch.empty(M_pad, packing.act_nbytes_per_row(N, fp4), dtype=torch.uint8, device=dev),
                        oscales=torch.empty(N // G, M_pad, dtype=torch.float8_e4m3fn if fp4 else torch.bfloat16, device=dev), lora_act_out=new(M_pad, 48, dtype=torch.float32))
            gemm_mod.svdq_gemm_w4a4(**kw, **outs, lora_down=nxt["proj_down"], smooth_factor=nxt["smooth_factor"])
        elif kind in ("rope", "split"):
            outs = dict(out=new(M, N)) if kind == "rope" else {k: new(1, N // 384, M_pad, 128, dtype=torch.float16) for k in ("out_q", "out_k", "out_v")}
            gemm_mod.svdq_gemm_w4a4(**kw, **outs, norm_q=nq, norm_k=nq, rotary_emb=rot, attn_tokens=M if kind == "split" else 0)
        else:
            outs = dict(out_linearattn=new(M_pad // 256, 256, N // 3), out_vk=new(M_pad // 256, N // 96, 33, 32, dtype=torch.float32))
            gemm_mod.svdq_gemm_w4a4(**kw, **outs)
        torch.cuda.synchronize()
        return outs

    if kind == "next":
        nxt = make_module(synth.make_layer(128, N, 48, seed=9, fp4=fp4), dev).native_tensors()
    if kind in ("rope", "split"):
        ang = 6.283 * torch.rand(M_pad, 64, generator=g)
        rot = packing.repack_rotemb(torch.stack((ang.sin(), ang.cos()), dim=-1).reshape(M_pad, 128).to(dev))
        nq = (1.0 + 0.2 * torch.randn(128, generator=g)).to(torch.bfloat16).to(dev)
    want, got, again = run(1), run(None), run(None)
    assert plans[0].few_rows == 0 and repr(plans[1]) == repr(plans[2])
    for name in got:
        a, b = got[name].cpu(), want[name].cpu()
        assert torch.equal(a.view(torch.uint8), again[name].cpu().view(torch.uint8)), f"{name} changed between two launches"
        if name == "qout":
            continue  # (checked through the codes below)
        a, b = a.float(), b.float()
        assert not torch.isnan(a).any(), name
        # sums of K products and R more in another order: 2^-24 (K + R) of the largest value at most; then, for the 16-bit
        # outputs, one rounding that may go the other way
        tol = (K + R) * 2.0**-24 * b.abs().max()
        if name in ("out_vk", "lora_act_out"):  # sums of bf16 values that may differ so: one in a hundred by an ulp (2^-8)
            assert (a - b).norm() <= 2.0**-8 * 0.1 * b.norm() + tol, name
        elif name == "oscales":
            assert ((a - b).abs() <= 2.0**-3 * b.abs()).all() and (a != b).float().mean() < 1e-2  # (an e4m3 step is an eighth at most)
        else:
            assert ((a - b).abs() <= torch.maximum(bf16_ulp(torch.maximum(a.abs(), b.abs())), tol)).all(), f"{name}: {(a - b).abs().max()}"
            assert (a != b).float().mean().item() < 2e-2, name
    if kind == "next":  # the codes belong to the bf16 tile stored next to them
        from oracle import quant

        nl = synth.make_layer(128, N, 48, seed=9, fp4=fp4)
        h = got["out"].cpu()
        codes, scales = quant.quantize_act_nvfp4(h, nl.smooth) if fp4 else quant.quantize_act_int4(h, nl.smooth, unsigned=True, shift=quant.SHIFT_GELU)
        logical = packing.act_to_logical(got["qout"].cpu(), N, fp4=fp4, unsigned=not fp4)
        assert torch.equal(logical.to(codes.dtype), codes)
        assert torch.equal(packing.scales_to_logical(got["oscales"].cpu(), fp4).view(torch.uint8), scales.view(torch.uint8))
    return plans[1]


@pytest.mark.parametrize("fp4", [False, True])
def test_all_rows_of_qout_whatever_M_out(dev, fp4):
    """``M_out`` and ``N_out`` are the shape of ``out``: a call of the C ABI that writes ``qout`` alone works out all M_pad rows,
    whatever they hold."""
    import ctypes

    from nunchaku_amd import _native as nv
    from nunchaku_amd import packing

    M, K, N, R, R2 = 512, 256, 384, 16, 32
    announce(f"qout without out, M_out set, fp4={fp4}")
    m, nxt = make_module(synth.make_layer(N, K, R, seed=3, fp4=fp4), dev), make_module(synth.make_layer(128, N, R2, seed=9, fp4=fp4), dev)
    t, n = m.native_tensors(), nxt.native_tensors()
    act, asc, la = m.quantize(synth.make_activations(M, K, seed=M).to(dev))

    def run(M_out):
        qout = torch.full((M, packing.act_nbytes_per_row(N, fp4)), 0xA5, dtype=torch.uint8, device=dev)
        osc = torch.full((N // (16 if fp4 else 64), M * (1 if fp4 else 2)), 0xA5, dtype=torch.uint8, device=dev)
        down = torch.full((M, R2), float("nan"), dtype=torch.float32, device=dev)
        a = nv.GemmArgs(act=act.data_ptr(), ascales=asc.data_ptr(), wgt=t["qweight"].data_ptr(), wscales=t["wscales"].data_ptr(),
                        colnorm=nv.ptr(t["wscales"].colnorm), bias=t["bias"].data_ptr(), wcscales=nv.ptr(t["wcscales"]), lora_act_in=la.data_ptr(),
                        lora_up=t["proj_up"].data_ptr(), qout=qout.data_ptr(), oscales=osc.data_ptr(), next_smooth_rcp=n["smooth_factor"].data_ptr(),
                        next_lora_down=n["proj_down"].data_ptr(), next_lora_act_out=down.data_ptr(), M_pad=M, N=N, K=K, M_out=M_out, R_up=R, R_down=R2,
                        alpha=m.alpha, fp4=int(fp4))
        nv.launch(nv.lib().svdq_gemm_w4a4, ctypes.byref(a), dev)
        torch.cuda.synchronize()
        return qout, osc, down

    want = run(0)
    assert not torch.isnan(want[2]).any()
    for M_out in (40, M, M + 1):
        for a, b in zip(run(M_out), want):
            assert torch.equal(a, b), M_out
