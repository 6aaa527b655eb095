"""The host extension (csrc/host_ext.cpp) takes the plain calls and hands every other one back to the Python path: both give
the same bits, and what the extension keeps of a layer never outlives a change of its parameters."""

import pytest
import torch

from conftest import announce
from gpu_util import make_module
from oracle import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp4", [False, True])
@pytest.mark.parametrize("M,R", [(1, 16), (257, 48)])
def test_linear_fast_and_checked_path(dev, M, R, fp4):
    from nunchaku_amd import _native as nv

    announce(f"host extension linear M={M} R={R} fp4={fp4}")
    K, N = 256, 384
    m = make_module(synth.make_layer(N, K, R, seed=M, fp4=fp4), dev)
    x = synth.make_activations(M, K, seed=M).to(dev).view(1, M, K)
    want = m._forward_by_operators(x[0], None)[:M]
    y = m(x)
    given = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    y2 = m(x, given)
    assert nv.host().linear(m._call.handle, m, x, None, 0, False) is not None, "the plain call is not taken by the extension"
    torch.cuda.synchronize()
    assert y.shape == (1, M, N) and torch.equal(y[0], want) and torch.equal(given, want) and y2.data_ptr() == given.data_ptr()
    # factors as a list (fast), and as a tuple (not the plain case)
    m.lora_scales = [0.5] * ((R + 15) // 16)
    scaled = m(x)
    m.lora_scales = tuple(m.lora_scales)
    assert nv.host().linear(m._call.handle, m, x, None, 0, False) is None
    assert torch.equal(m(x), scaled) and not torch.equal(scaled, y)
    m.lora_scales = None
    # a parameter written to in place, and one replaced: the kept handle is not used any more
    with torch.no_grad():
        m.proj_up.mul_(2.0)
    assert nv.host().linear(m._call.handle, m, x, None, 0, False) is None
    twice = m(x)
    m.proj_up = torch.nn.Parameter(m.proj_up.detach() * 0.5, requires_grad=False)
    torch.cuda.synchronize()
    assert not torch.equal(twice, y) and torch.equal(m(x), y)
    with pytest.raises(RuntimeError):  # (view of a tensor that is not contiguous)
        m(x.expand(2, M, K).transpose(1, 2))
    with pytest.raises(ValueError):
        m(x[:, :, :128].contiguous())
    with pytest.raises(NotImplementedError):
        m(x.to(torch.float16))
    with pytest.raises(ValueError):
        m(x, torch.empty(M, N - 8, dtype=torch.bfloat16, device=dev))


@pytest.mark.parametrize("M,pad", [(5, 256), (300, 512)])
def test_mlp_and_awq_fast_and_checked_path(dev, M, pad, monkeypatch):
    from nunchaku_amd import _native as nv
    from nunchaku_amd.models import AWQW4A16Linear
    from nunchaku_amd.ops import fused_gelu_mlp

    announce(f"host extension mlp M={M} pad={pad}, awq")
    m1 = make_module(synth.make_layer(512, 256, 32, seed=1), dev)
    m2 = make_module(synth.make_layer(256, 512, 32, seed=2), dev, act_unsigned=True)
    x = synth.make_activations(M, 256, seed=M).to(dev).view(1, M, 256)
    awq = AWQW4A16Linear(128, 64, device=dev)
    g = torch.Generator().manual_seed(3)
    awq.load_state_dict(dict(qweight=torch.randint(-2**31, 2**31 - 1, (16, 64), generator=g, dtype=torch.int32), wscales=0.01 * torch.rand(2, 64, generator=g).bfloat16(),
                             wzeros=-0.05 * torch.rand(2, 64, generator=g).bfloat16(), bias=torch.randn(64, generator=g).bfloat16()))
    v = torch.randn(2, 3, 128, generator=g).bfloat16().to(dev)
    y, z = fused_gelu_mlp(x, m1, m2, pad_size=pad), awq(v)
    assert y.shape == (1, M, 256) and z.shape == (2, 3, 64)

    class Declines:  # every call goes to the checked path
        make_layer = staticmethod(nv.host().make_layer)

        def __getattr__(self, name):
            return lambda *args: None

    monkeypatch.setattr(nv, "_host_module", Declines())
    assert torch.equal(fused_gelu_mlp(x, m1, m2, pad_size=pad), y) and torch.equal(awq(v), z)


def test_arguments_outside_the_plain_case(dev):
    """A rank above the largest one (its factors would not fit the extension's array) and numbers that are not whole are
    refused as the checked path refuses them."""
    from nunchaku_amd.models.linear import SVDQW4A4Linear
    from nunchaku_amd.ops import fused_gelu_mlp

    announce("host extension: rank 1040, pad_size 256.0")
    m = SVDQW4A4Linear(256, 384, rank=1040, device=dev)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_(torch.ones(p.shape, dtype=p.dtype, device=dev))
    x = synth.make_activations(16, 256, seed=1).to(dev).view(1, 16, 256)
    m.lora_scales = [1.0] * 65
    for _ in range(2):  # the call that converts the layer and the one behind it
        with pytest.raises(ValueError, match="rank"):
            m(x)
    m1 = make_module(synth.make_layer(512, 256, 32, seed=1), dev)
    m2 = make_module(synth.make_layer(256, 512, 32, seed=2), dev, act_unsigned=True)
    fused_gelu_mlp(x, m1, m2)
    with pytest.raises(TypeError):
        fused_gelu_mlp(x, m1, m2, pad_size=256.0)


def test_a_true_NO_ALLOC_of_any_type(dev, monkeypatch):
    """``NO_ALLOC = 1`` selects the fixed scratch as ``True`` does, through every call of the extension: a split that does not
    fit it is refused."""
    from nunchaku_amd import packing
    from nunchaku_amd.ops import fused_gelu_mlp, fused_qkv_norm_rottary
    from nunchaku_amd.ops import gemm as gemm_mod

    announce("host extension: NO_ALLOC = 1")
    m1 = make_module(synth.make_layer(2048, 1024, 16, seed=1), dev)
    m2 = make_module(synth.make_layer(1024, 2048, 16, seed=2), dev, act_unsigned=True)
    x = synth.make_activations(2048, 1024, seed=1).to(dev).view(1, 2048, 1024)
    m3 = make_module(synth.make_layer(2304, 1024, 16, seed=3), dev)
    norm = torch.nn.RMSNorm(128, device=dev, dtype=torch.bfloat16)
    rot = packing.repack_rotemb(torch.zeros(2048, 128, device=dev))
    m1(x), fused_gelu_mlp(x, m1, m2), fused_qkv_norm_rottary(x, m3, norm, norm, rot)
    monkeypatch.setattr(gemm_mod, "K_SPLIT", 16)  # 128 tiles and more x 16 parts x 128 KB
    for value in (True, 1):
        monkeypatch.setattr(gemm_mod, "NO_ALLOC", value)
        with pytest.raises(NotImplementedError, match="fixed scratch"):
            m1(x)
        with pytest.raises(NotImplementedError, match="fixed scratch"):
            fused_gelu_mlp(x, m1, m2)
        with pytest.raises(NotImplementedError, match="fixed scratch"):
            fused_qkv_norm_rottary(x, m3, norm, norm, rot)


@pytest.mark.parametrize("R,fp4", [(0, False), (48, False), (48, True)])
def test_operators_fast_and_checked_path(dev, R, fp4, monkeypatch):
    """Each operator hands the library the same argument block, and refuses the same calls with the same words, whether the
    extension fills the block in or the Python code does."""
    from nunchaku_amd import _native as nv
    from nunchaku_amd import packing
    from nunchaku_amd.ops import gemm as gemm_mod
    from nunchaku_amd.ops import linearattn_vk_mul_q, svdq_gemm_w4a4, svdq_quantize_w4a4_act_fuse_lora

    announce(f"host extension: operators R={R} fp4={fp4}")
    M, K, N = 300, 256, 384
    t = make_module(synth.make_layer(N, K, R, seed=M, fp4=fp4), dev).native_tensors()
    x = synth.make_activations(M, K, seed=M).to(dev)
    act, asc, la = svdq_quantize_w4a4_act_fuse_lora(x, lora_down=t["proj_down"], smooth=t["smooth_factor"], fp4=fp4)
    host, real_launch = nv.host(), nv.launch
    taken, blocks = [], []

    class Host:
        def __init__(self, declines):
            self.declines = declines

        def __getattr__(self, name):
            def call(*args):
                r = None if self.declines else getattr(host, name)(*args)
                taken.append(r is not None)
                return r

            return call

    def launch(entry, ref, device):  # (no kernel: what it would be given.  Where a result lies that the call itself allocates is the allocator's choice)
        a = ref._obj
        own = ("output", "oscales", "lora_act_out") if isinstance(a, nv.QuantizeArgs) else ("lora_scales", "qkv_head_stride", "norm_eps")  # (read with a rotary table only)
        fields = (nv.QuantizeArgs if isinstance(a, nv.QuantizeArgs) else nv.GemmArgs)._fields_
        block = {n: getattr(a, n) for n, _ in fields if n not in own}
        if isinstance(a, nv.GemmArgs):
            block["lora_scales"] = [a.lora_scales[i] for i in range((a.R_up + 15) // 16)]
        blocks.append((entry is nv.lib().svdq_gemm_w4a4_noalloc, block))

    monkeypatch.setattr(nv, "launch", launch)

    def run(declines, f, kw):
        monkeypatch.setattr(nv, "_host_module", Host(declines))
        blocks.clear(), taken.clear()
        try:
            r = f(**kw)
            shapes = [(tuple(o.shape), o.dtype, o.is_contiguous()) for o in r] if isinstance(r, tuple) else None
            return shapes, list(blocks), list(taken)
        except Exception as e:
            return (type(e), str(e)), None, list(taken)

    def same(f, plain, **kw):
        fast, checked = run(False, f, kw), run(True, f, kw)
        assert fast[:2] == checked[:2] and fast[2] == [plain], (f.__name__, {k: v for k, v in kw.items() if not isinstance(v, torch.Tensor)}, fast, checked)

    quant = lambda plain, **kw: same(svdq_quantize_w4a4_act_fuse_lora, plain, **{**dict(input=x, lora_down=t["proj_down"], smooth=t["smooth_factor"], fp4=fp4), **kw})
    quant(True)
    quant(True, smooth=None, pad_size=512, input=x[:1])
    for kw in (dict(pad_size=128), dict(input=x.half()), dict(input=x[0]), dict(input=x[:, :128]), dict(input=x.T.contiguous().T), dict(smooth=t["smooth_factor"][:128]), dict(lora_down=None), dict(input=x[:0]), dict(input=x.cpu())):
        fast, checked = (run(d, svdq_quantize_w4a4_act_fuse_lora, {**dict(input=x, lora_down=t["proj_down"], smooth=t["smooth_factor"], fp4=fp4), **kw}) for d in (False, True))
        assert fast[:2] == checked[:2] and not any(fast[2]), (kw.keys(), fast, checked)

    out = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    q, vk = torch.empty(2, 256, N // 3, dtype=torch.bfloat16, device=dev), torch.empty(2, N // 96, 33, 32, device=dev)
    base = dict(act=act, wgt=t["qweight"], out=out, ascales=asc, wscales=t["wscales"], lora_act_in=la, lora_up=t["proj_up"], bias=t["bias"], wcscales=t["wcscales"], fp4=fp4)
    lowrank = R > 0  # (an empty low-rank branch is not the plain case)
    gemm = lambda plain, **kw: same(svdq_gemm_w4a4, plain, **{**base, **kw})
    gemm(lowrank)
    gemm(True, lora_act_in=None, lora_up=None, bias=None, alpha=0.25)
    gemm(lowrank, act_unsigned=True, fuse_silu=True, out=out[:, :100].contiguous())
    gemm(lowrank, lora_scales=[0.5, 2.0], out=out.view(1, M, N))
    gemm(lowrank, lora_scales=[0.5] * 9)
    gemm(False, lora_scales=(0.5, 1, 2))
    gemm(False, alpha=torch.tensor(0.5))
    gemm(lowrank, out=None, out_vk=vk, out_linearattn=q)
    for split, no_alloc in ((3, False), (None, 1)):
        monkeypatch.setattr(gemm_mod, "K_SPLIT", split), monkeypatch.setattr(gemm_mod, "NO_ALLOC", no_alloc)
        gemm(lowrank)
    for kw in (dict(act=None), dict(wgt=None), dict(act=act[:, :-16].contiguous()), dict(act=act[:128]), dict(ascales=asc[:-1]), dict(ascales=asc.view(torch.uint8)), dict(out=None),
               dict(lora_up=None), dict(lora_act_in=la[:256]), dict(bias=t["bias"][:-1]), dict(out=out.half()), dict(out=out.T), dict(out=out.cpu()), dict(act=act.cpu()),
               dict(out_vk=vk), dict(out=None, out_vk=vk, out_linearattn=q, fuse_silu=True), dict(out=None, out_vk=vk[:1], out_linearattn=q), dict(out=None, out_vk=vk.half(), out_linearattn=q),
               dict(out=None, out_vk=vk, out_linearattn=q[:1]), dict(poolout=out), dict(norm_q=t["bias"]), dict(lora_down=t["proj_down"])):
        fast, checked = run(False, svdq_gemm_w4a4, {**base, **kw}), run(True, svdq_gemm_w4a4, {**base, **kw})
        assert fast[:2] == checked[:2] and (isinstance(fast[0], tuple) or not lowrank) and not any(fast[2]), (kw.keys(), fast, checked)

    monkeypatch.setattr(nv, "launch", real_launch)
    vk.uniform_(0.5, 1.0)
    x3 = torch.rand(2, 256, N // 3, device=dev).bfloat16()
    for tokens in (None, 77):
        got = []
        for declines in (False, True):
            monkeypatch.setattr(nv, "_host_module", Host(declines))
            got.append(linearattn_vk_mul_q(x3.clone(), vk, tokens))
        assert torch.equal(*got)
    for args in ((x3, vk, 257), (x3, vk, 0), (x3[:1], vk), (x3.half(), vk), (x3, vk.cpu()), (x3.transpose(0, 1), vk), (x3.cpu(), vk)):
        seen = []
        for declines in (False, True):
            monkeypatch.setattr(nv, "_host_module", Host(declines))
            with pytest.raises((ValueError, RuntimeError)) as e:
                linearattn_vk_mul_q(*args)
            seen.append((type(e.value), str(e.value)))
        assert seen[0] == seen[1], seen
