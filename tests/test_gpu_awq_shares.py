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
