"""The projecting workgroups of the few-rows quantize kernel (csrc/quantize.hip, ``project_rows``): every number of chunks that a wave
can have against the chunks it keeps on their way (three with one rank tile, one with two), waves with one chunk less than others and
with none."""

import pytest

from conftest import announce
from test_gpu_quantize import _check_row_sample, _run
from oracle import linear as olin
from oracle import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [1, 7, 8, 9, 16, 23, 24, 25, 32, 33, 40, 49, 57, 65, 72])
@pytest.mark.parametrize("M,R", [(40, 32), (900, 80)])  # one rank tile per projecting workgroup; two, and one left over
def test_chunks_per_wave(dev, M, R, chunks):
    announce(f"projection ring M={M} R={R} chunks={chunks}")
    K = 128 * chunks
    if M >= 512:
        return _check_row_sample(dev, M, K, R, False, True)
    layer = synth.make_layer(128, K, R, seed=chunks)
    x = synth.make_activations(M, K, seed=chunks)
    _, _, la = _run(dev, x, layer, fp4=False, smooth=True)
    want = olin.quantize_act_fuse_lora(x, layer.proj_down, layer.smooth)[2]
    assert (la - want).abs().max().item() <= 2e-5 * want.abs().max().item() + 1e-6  # (fp32 sums of K products in another order)


@pytest.mark.parametrize("M,K,R,fp4", [(2304, 640, 16, True), (2100, 1152, 64, False), (3072, 3200, 48, False), (4600, 384, 32, True), (4600, 3072, 32, True), (4096, 1152, 128, False),
                                       (6000, 640, 112, True), (1000, 9344, 16, False)])
def test_quantizing_and_projecting_apart_beyond_8_rows_per_compute_unit(dev, M, K, R, fp4):
    """One and two shares of the quantizing, one and two rank tiles per projecting workgroup, a rank tile left over, rows and chunks
    that end early; long rows with fewer chunks on their way."""
    announce(f"apart M={M} K={K} R={R} fp4={fp4}")
    _check_row_sample(dev, M, K, R, fp4, True)


@pytest.mark.parametrize("K,R,fp4,apart,together", [(1152, 64, False, 2304, 4608), (640, 112, True, 2304, 9216), (1152, 48, True, 3072, 9216),
                                                     (1152, 32, False, 2048, 4096), (6272, 32, True, 2048, 4096)])
def test_projections_keep_their_bits_from_form_to_form(dev, K, R, fp4, apart, together):
    """On either side of the most rows for which quantizing and projecting go apart a row's projection is the same: the sums of the waves are added in one
    order.  (It does change, on 256 compute units, for NVFP4 at ranks 80 ... 128 from 2048 rows to more and at rank 32, K <= 6144, from 4096 to more, where
    eight waves become four, and beyond 8192 rows for INT4 at ranks 80 ... 128, where the rows are split.)"""
    from gpu_util import make_module

    announce(f"projection bits K={K} R={R} fp4={fp4}")
    m = make_module(synth.make_layer(128, K, R, seed=R, fp4=fp4), dev)
    x = synth.make_activations(max(apart, together), K, seed=K).to(dev)
    n = min(apart, together)
    assert m.quantize(x[:apart])[2][:n].equal(m.quantize(x[:together])[2][:n])
