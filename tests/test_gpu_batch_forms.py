"""GPU parity of every form of the batch kernels, bit for bit against the oracle.
Each case names the form that the dispatch gives it (vtq.probe.form).
"""
import pytest

import vtq
from vtq import probe, synth

from test_gpu_parity import check

pytestmark = pytest.mark.gpu

INT = vtq.REGIME_INTEGER


# Q4_K batches below 32 rows on grids past those of short rows and small matrices
@pytest.mark.parametrize("batch,in_f,out_f,form", [(5, 17 * 256, 8200, 304), (31, 17 * 256, 8161, 304), (4, 127 * 256, 8165, 316),
                                                   (8, 256, 33000, probe.PER_WAVE), (20, 768, 32801, probe.PER_WAVE),
                                                   (4, 2048, 33000, probe.GEMV)])
def test_q4k_small_batches_on_large_matrices(ctx, batch, in_f, out_f, form):
    assert probe.form(vtq.Q4_K, INT, batch, in_f, out_f) == form
    w = synth.weights(vtq.Q4_K, out_f, in_f, seed=in_f + out_f)
    check(ctx, vtq.Q4_K, INT, synth.activations(batch * in_f, seed=in_f + batch), w, batch, in_f, out_f)


# Q6_K batches of 3 to 7 rows either side of their line
@pytest.mark.parametrize("batch,in_f,out_f,form", [(3, 4096, 4097, 302), (3, 4096, 4095, probe.GEMV), (4, 43 * 256, 1050, 304),
                                                   (5, 32 * 256, 1400, probe.GEMV), (7, 256, 32769, 301)])
def test_q6k_small_batches(ctx, batch, in_f, out_f, form):
    assert probe.form(vtq.Q6_K, INT, batch, in_f, out_f) == form
    w = synth.weights(vtq.Q6_K, out_f, in_f, seed=in_f + out_f)
    check(ctx, vtq.Q6_K, INT, synth.activations(batch * in_f, seed=in_f + batch), w, batch, in_f, out_f)
