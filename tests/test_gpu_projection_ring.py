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
