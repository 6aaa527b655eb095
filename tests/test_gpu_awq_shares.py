"""The AWQ GEMV with one workgroup per compute unit: shares of the channels that end inside a tile of 16, on either side of one, two and
several tiles per workgroup (256 compute units), the last share the shortest.  Bound: one rounding to bf16, and fp32 sums of ic terms."""

import pytest
import torch

from conftest import announce
from oracle import awq
from test_gpu_awq import _module

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 8])
@pytest.mark.parametrize("oc,ic", [(16, 640), (20, 1088), (4092, 640), (4100, 640), (8196, 1088), (9220, 640), (18432, 640), (24572, 640)])
def test_shares_that_end_inside_a_tile(dev, rows, oc, ic):
    announce(f"awq gemv rows={rows} oc={oc} ic={ic} (shares)")
    m, (codes, scales, zeros, _) = _module(dev, oc, ic, seed=oc + ic, bias=False)
    x = torch.randn(rows, ic, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    y = m(x.to(dev)).double().cpu()
    w = awq.dequant(codes, scales, zeros).double()
    want = x.double() @ w.T
    assert ((y - want).abs() <= 2.0**-8 * want.abs() + ic * 2.0**-24 * (x.double().abs() @ w.abs().T)).all()


@pytest.mark.parametrize("rows,oc,ic", [(1, 18432, 640), (8, 9220, 640), (5, 20, 1088), (3, 28676, 128)])
def test_scales_and_zeros_off_a_word(dev, rows, oc, ic):
    """Scales and zeros need the alignment of a bf16 value only: 2 bytes off a word they give the same bits (the last shape has a
    workgroup per tile)."""
    from nunchaku_amd.ops.gemv import awq_gemv_w4a16

    announce(f"awq gemv rows={rows} oc={oc} ic={ic} (scales off a word)")
    m, _ = _module(dev, oc, ic, seed=rows, bias=False)
    x = torch.randn(rows, ic, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16).to(dev)

    def off(t):
        raw = torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)
        raw[1:].copy_(t.reshape(-1))
        assert raw[1:].data_ptr() % 4 == 2
        return raw[1:].view(t.shape)

    y = awq_gemv_w4a16(x, m.qweight, m.wscales, m.wzeros, rows, oc, ic)
    assert torch.equal(awq_gemv_w4a16(x, m.qweight, off(m.wscales), off(m.wzeros), rows, oc, ic), y)
