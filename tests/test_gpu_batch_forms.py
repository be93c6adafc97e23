"""GPU parity of the k-quant batch kernels where the dispatch changes form, and of
all of them with y aligned to 4 bytes; bit for bit against the oracle.  Each case
names the form that the dispatch gives it (vtq.probe.form).
"""
import pytest

import oracle as O
import vtq
from vtq import probe, synth

from test_gpu_parity import THREADS, assert_bits_equal, check

pytestmark = pytest.mark.gpu

INT = vtq.REGIME_INTEGER


# Q4_K batches below 32 rows on grids past those of short rows and small matrices,
# and the larger pieces of long rows
@pytest.mark.parametrize("batch,in_f,out_f,form", [(5, 17 * 256, 8200, 304), (31, 17 * 256, 8161, 304), (4, 127 * 256, 8165, 316),
                                                   (8, 256, 33000, probe.PER_WAVE), (20, 768, 32801, probe.PER_WAVE),
                                                   (4, 2048, 33000, probe.GEMV), (16, 64 * 256, 40, 308),
                                                   (16, 126 * 256, 40, 316)])
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


# y aligned to 4 bytes only: rows whose length is a multiple of 4 are stored 16 bytes at a time
@pytest.mark.parametrize("t,regime,batch,in_f,out_f,form", [
    (vtq.Q4_K, INT, 40, 17 * 256, 8192, probe.LDS_OPERAND), (vtq.Q4_K, INT, 33, 256, 33000, probe.PER_WAVE),
    (vtq.Q4_K, INT, 9, 4096, 1028, 302), (vtq.Q6_K, INT, 9, 2048, 132, 301), (vtq.Q6_K, INT, 65, 512, 12004, 604),
    (vtq.Q8_0, INT, 150, 992, 300, 14), (vtq.Q8_0, INT, 193, 160, 4472, 21)])
def test_y_aligned_to_4_bytes(ctx, t, regime, batch, in_f, out_f, form):
    import torch

    assert probe.form(t, regime, batch, in_f, out_f) == form
    w, x = synth.weights(t, out_f, in_f, seed=out_f), synth.activations(batch * in_f, seed=batch)
    dx, dw = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    want = O.linear_dispatch(t, regime, x, w, batch, in_f, out_f, THREADS)
    for shift in (1, 2, 3):
        buf = torch.full((batch * out_f + 8,), 7.0, device="cuda")
        y = buf[shift:shift + batch * out_f]
        ctx.linear_device(t, regime, dx.data_ptr(), dw.data_ptr(), dw.numel(), y.data_ptr(), batch, in_f, out_f, None)
        torch.cuda.synchronize()
        assert_bits_equal(y.cpu().numpy(), want, f"shift {shift}")
        assert bool((buf[:shift] == 7.0).all()) and bool((buf[shift + batch * out_f:] == 7.0).all())
