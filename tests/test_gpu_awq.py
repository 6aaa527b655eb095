"""AWQ W4A16 GEMV on the GPU against the oracle: the module with the reference's parameter layout, every
row count 1..8, ragged K (not a multiple of 512), the Qwen-Image modulation shape, and linearity."""

import numpy as np
import pytest
import torch

from conftest import announce
from oracle import awq

pytestmark = pytest.mark.gpu


def _module(dev, oc, ic, seed, bias=True):
    from nunchaku_amd.models import AWQW4A16Linear

    codes, scales, zeros, b = awq.make_layer(oc, ic, seed)
    m = AWQW4A16Linear(ic, oc, bias=bias, device=dev)
    sd = {"qweight": torch.from_numpy(awq.pack_w4(codes.numpy()).view(np.int32).copy()), "wscales": scales, "wzeros": zeros}
    if bias:
        sd["bias"] = b
    m.load_state_dict(sd, strict=True)
    return m, (codes, scales, zeros, b if bias else None)


def _check(y, want, bias):
    """fp32 accumulation in another order, then the bf16 rounding(s) of the reference: within one bf16 ulp of
    the oracle rounded the same way, and rel-L2 1e-3."""
    want_bf = want.to(torch.bfloat16).float()
    if bias is not None:
        want_bf = (want_bf + bias.float()).to(torch.bfloat16).float()
    got = y.float().cpu()
    rel = ((got - want_bf).norm() / want_bf.norm()).item()
    assert rel <= 1e-3, f"rel-L2 {rel:.3e}"
    ulp = torch.pow(2.0, torch.floor(torch.log2(want_bf.abs().clamp_min(2.0**-126))) - 7)
    assert ((got - want_bf).abs() <= 2 * ulp + 1e-6).all()


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("oc,ic", [(256, 512), (64, 192), (520, 1088)])
def test_against_oracle(dev, rows, oc, ic):
    announce(f"awq gemv rows={rows} oc={oc} ic={ic}")
    m, (codes, scales, zeros, bias) = _module(dev, oc, ic, seed=oc + ic)
    x = torch.randn(rows, ic, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    y = m(x.to(dev))
    torch.cuda.synchronize()
    assert y.shape == (rows, oc) and y.dtype == torch.bfloat16
    _check(y, awq.gemv(x, codes, scales, zeros), bias)


@pytest.mark.parametrize("rows", [1, 5, 8])
@pytest.mark.parametrize("oc,ic", [(16, 64), (20, 128), (12, 192), (100, 2112), (52, 4096), (28676, 128)])
def test_edges_of_the_tile_walk(dev, rows, oc, ic):
    """A last tile that begins early (oc not a multiple of 16), fewer channels than a tile, one to four steps of K per wave
    with and without a remainder, and many channels with short rows (a workgroup per tile)."""
    announce(f"awq gemv rows={rows} oc={oc} ic={ic}")
    m, (codes, scales, zeros, bias) = _module(dev, oc, ic, seed=oc + ic)
    x = torch.randn(rows, ic, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    y = m(x.to(dev))
    torch.cuda.synchronize()
    _check(y, awq.gemv(x, codes, scales, zeros), bias)


@pytest.mark.parametrize("rows", [1, 5, 8])
@pytest.mark.parametrize("oc,ic", [(28676, 640), (16384, 512), (16388, 512)])
def test_many_channels(dev, rows, oc, ic):
    """More tiles per workgroup than meet at once, and either side of the line behind which short rows have a workgroup per tile.
    Bound: one rounding to bf16, and fp32 sums of ic terms."""
    announce(f"awq gemv rows={rows} oc={oc} ic={ic} (many channels)")
    m, (codes, scales, zeros, _) = _module(dev, oc, ic, seed=oc + ic, bias=False)
    x = torch.randn(rows, ic, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    y = m(x.to(dev)).double().cpu()
    w = awq.dequant(codes, scales, zeros).double()
    want = x.double() @ w.T
    assert ((y - want).abs() <= 2.0**-8 * want.abs() + ic * 2.0**-24 * (x.double().abs() @ w.abs().T)).all()


def test_long_k_takes_the_path_without_lds_staging(dev):
    """8 rows of K=4160 do not fit the 64 KB the kernel stages x in: the activations then come from global memory."""
    oc, ic, rows = 64, 4160, 8
    announce(f"awq gemv rows={rows} oc={oc} ic={ic} (x not staged)")
    m, (codes, scales, zeros, bias) = _module(dev, oc, ic, seed=77)
    x = torch.randn(rows, ic, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    y = m(x.to(dev))
    torch.cuda.synchronize()
    _check(y, awq.gemv(x, codes, scales, zeros), bias)
    _check(m(x[:1].to(dev)), awq.gemv(x[:1], codes, scales, zeros), bias)  # one row of the same layer: staged


def test_modulation_shape_and_linearity(dev):
    """K=3072, N=18432 (six modulation vectors of a 3072-wide block), one row; without bias the result is
    linear in x up to the bf16 rounding of the output."""
    oc, ic = 18432, 3072
    announce(f"awq gemv modulation shape oc={oc} ic={ic}")
    m, (codes, scales, zeros, _) = _module(dev, oc, ic, seed=9, bias=False)
    x = torch.randn(1, 1, ic, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    y = m(x.to(dev))
    torch.cuda.synchronize()
    assert y.shape == (1, 1, oc)
    _check(y[0], awq.gemv(x[0], codes, scales, zeros), None)
    y2 = m((x * 2).to(dev))  # doubling is exact in bf16
    assert torch.equal(y2.float(), y.float() * 2)


def test_rejects_bad_arguments(dev):
    from nunchaku_amd.ops import awq_gemv_w4a16_cuda

    m, _ = _module(dev, 64, 128, seed=1)
    x = torch.zeros(9, 128, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):  # more than 8 rows
        m(x)
    with pytest.raises(NotImplementedError):
        awq_gemv_w4a16_cuda(x[:1], m.qweight, m.wscales, m.wzeros, 1, 64, 128, group_size=128)
    with pytest.raises(RuntimeError, match="GPU"):
        awq_gemv_w4a16_cuda(x[:1].cpu(), m.qweight, m.wscales, m.wzeros, 1, 64, 128)


def test_bias_wherever_the_module_keeps_it(dev):
    """The bias is what ``module.bias`` gives: a parameter, a tensor assigned to a layer built without one, a buffer, a
    parametrization, a class attribute."""
    from torch import nn
    from torch.nn.utils import parametrize

    from nunchaku_amd.models import AWQW4A16Linear
    from nunchaku_amd.ops import awq_gemv_w4a16_cuda

    oc, ic = 64, 128
    announce("awq layer with its bias in other places than its parameters")
    g = torch.Generator().manual_seed(1)
    x = torch.randn(2, ic, generator=g).to(torch.bfloat16).to(dev)
    bias = torch.randn(oc, generator=g).to(torch.bfloat16).to(dev)

    def want(m, b):
        return awq_gemv_w4a16_cuda(x, m.qweight, m.wscales, m.wzeros, 2, oc, ic, 64, b)

    m, _ = _module(dev, oc, ic, seed=1, bias=False)
    assert torch.equal(m(x), want(m, None)) and not torch.equal(want(m, bias), want(m, None))
    m.bias = bias
    assert torch.equal(m(x), want(m, bias))
    del m.bias
    m.register_buffer("bias", bias)
    assert torch.equal(m(x), want(m, bias))

    class Twice(nn.Module):
        def forward(self, b):
            return b * 2

    m, _ = _module(dev, oc, ic, seed=1)
    parametrize.register_parametrization(m, "bias", Twice())
    assert torch.equal(m(x), want(m, m.bias.detach())) and not torch.equal(m(x), want(m, m.parametrizations.bias.original.detach()))

    class WithClassBias(AWQW4A16Linear):
        pass

    m, _ = _module(dev, oc, ic, seed=1, bias=False)
    del m.bias
    m.__class__ = WithClassBias
    WithClassBias.bias = bias
    assert torch.equal(m(x), want(m, bias))


@pytest.mark.parametrize("K", [64, 192, 1088, 4160])
def test_scales_and_zeros_up_to_infinity(dev, K):
    """A scale near the top of bf16's range and an infinite zero in the last group of channels, at lengths of K that end inside a
    step of 128 channels and leave waves without a step: each only reaches the outputs of its own channel, and there gives
    what the weights bf16(code * scale + zero) give."""
    from nunchaku_amd.ops import awq_gemv_w4a16_cuda

    N, M = 64, 3
    announce(f"awq gemv with extreme scales and zeros K={K}")
    g = torch.Generator().manual_seed(K)
    codes = torch.randint(0, 16, (N, K), generator=g)
    scales = (0.5 + torch.rand(K // 64, N, generator=g)).to(torch.bfloat16)
    zeros = (torch.randint(-16, 17, (K // 64, N), generator=g) / 8).to(torch.bfloat16)  # (sums with code * scale are exact in fp32)
    scales[-1, 5], zeros[-1, 5] = 2.0**120, 0.0
    scales[0, 21] = 2.0**123
    zeros[-1, 9], zeros[-1, 40] = float("inf"), float("-inf")
    x = (2.0**-20 * (0.5 + torch.rand(M, K, generator=g))).to(torch.bfloat16)  # (positive: an infinite weight gives infinity)
    qweight = torch.from_numpy(awq.pack_w4(codes.numpy()).view(np.int32).copy())
    out = awq_gemv_w4a16_cuda(x.to(dev), qweight.to(dev), scales.to(dev), zeros.to(dev), M, N, K).cpu()
    w = awq.dequant(codes, scales, zeros)
    want = x.double() @ w.double().T
    finite = torch.isfinite(want)
    assert (~finite).sum() == 2 * M and torch.equal(out[~finite].double(), want[~finite])
    # one rounding to bf16 and fp32 sums of K positive and negative terms
    bound = 2.0**-8 * want.abs() + K * 2.0**-24 * (x.double() @ w.double().abs().T)
    assert ((out.double() - want).abs() <= bound)[finite].all()
