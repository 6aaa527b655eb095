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
