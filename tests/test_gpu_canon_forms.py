"""Every form of the batched pinned dot (canon_gemm.hip, canon_gemm_split.hip),
every format, with rows of one, two and three 8192-input chunks and with edge
values.  Each case asserts the form that the dispatch gives it.  All outputs are
compared with batch-1 calls of the GEMV, and the outputs of some weight rows (the
first and last tiles and every 61st row) with the oracle.
"""
import numpy as np
import pytest

import oracle as O
import vtq
from vtq import probe, synth

from test_gpu_parity import F, THREADS, assert_bits_equal

pytestmark = pytest.mark.gpu

INT, FLOAT = vtq.REGIME_INTEGER, vtq.REGIME_FLOAT_FUSED
FORMATS = {"q8_0": (vtq.Q8_0, INT), "q5_0": (vtq.Q5_0, INT), "q4_0": (vtq.Q4_0, INT), "f32": (vtq.F32, INT),
           "q4_k": (vtq.Q4_K, FLOAT)}
# (tokens, outputs) of each form: 10 * token tiles of a wave + waves to a tile
SHAPES = {14: (33, 1300), 12: (50, 5210), 11: (97, 3530), 21: (193, 4470)}
# row lengths of one, two and three chunks, the last of several steps and a remainder
LENGTHS = {1: {"f32": 1001, "q4_k": 1280}, 2: {"f32": 8197 + 64, "q4_k": 8448}, 3: {"f32": 16451, "q4_k": 16640}}
BLOCK_LENGTHS = {1: 992, 2: 8224 + 64, 3: 16480}


def length(fmt, chunks):
    return LENGTHS[chunks].get(fmt, BLOCK_LENGTHS[chunks])


def weights(fmt, out_f, in_f, seed):
    if fmt == "f32":
        return np.random.default_rng(seed).standard_normal(out_f * in_f, F).view(np.uint8)
    return synth.weights(FORMATS[fmt][0], out_f, in_f, seed=seed)


def compare(ctx, fmt, form, x, w, in_f):
    import torch

    t, regime = FORMATS[fmt]
    batch, out_f = SHAPES[form]
    assert probe.form(t, regime, batch, in_f, out_f) == form
    print(f"[gpu] {fmt} form {form} {batch}x{in_f}->{out_f}", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    dx, dw = torch.from_numpy(x).cuda(), torch.cat([torch.from_numpy(w), torch.zeros(16, dtype=torch.uint8)]).cuda()
    y = torch.full((batch, out_f), float("nan"), device="cuda")
    ctx.linear_device(t, regime, dx.data_ptr(), dw.data_ptr(), w.size, y.data_ptr(), batch, in_f, out_f, stream)
    rows = torch.zeros(batch, (in_f + 3) // 4 * 4, device="cuda")  # each on 16 bytes
    rows[:, :in_f] = dx.view(batch, in_f)
    one = torch.full((batch, out_f), float("nan"), device="cuda")
    for b in range(batch):
        ctx.linear_device(t, regime, rows[b].data_ptr(), dw.data_ptr(), w.size, one[b].data_ptr(), 1, in_f, out_f, stream)
    got = y.cpu().numpy()
    assert_bits_equal(got, one.cpu().numpy(), "batch-1 calls")
    sel = np.unique(np.r_[0:40, 0:out_f:61, out_f - 40:out_f])
    ws = np.ascontiguousarray(w.reshape(out_f, -1)[sel]).reshape(-1)
    want = O.linear_dispatch(t, regime, x, ws, batch, in_f, sel.size, THREADS)
    assert_bits_equal(np.ascontiguousarray(got[:, sel]), want, "oracle")


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("form", SHAPES)
@pytest.mark.parametrize("chunks", [1, 2, 3])
def test_forms(ctx, fmt, form, chunks):
    in_f, (batch, out_f) = length(fmt, chunks), SHAPES[form]
    x = synth.activations(batch * in_f, seed=form + chunks)
    compare(ctx, fmt, form, x, weights(fmt, out_f, in_f, 3 * form + chunks), in_f)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("form", SHAPES)
def test_edge_values(ctx, fmt, form):
    # tokens of zeros, of one NaN or infinity at a row's first and last input
    # (the neighbouring tokens must not see them), of products in and below the
    # subnormal range, of sums that overflow
    in_f, (batch, out_f) = length(fmt, 1), SHAPES[form]
    x = synth.activations(batch * in_f, seed=17).reshape(batch, in_f)
    x[0], x[1] = 0.0, -0.0
    x[3, 0], x[5, -1], x[7, 0], x[9, -1] = np.nan, np.nan, np.inf, -np.inf
    x[10:16] *= F(1e-38)
    x[16:22] = (x[16:22] * F(1e-38) * F(1e-6)).astype(F)
    x[22:28] *= F(3e37)
    x[batch - 1, -1] = np.inf
    compare(ctx, fmt, form, x.reshape(-1), weights(fmt, out_f, in_f, 23), in_f)


@pytest.mark.parametrize("fmt", ["q8_0", "q5_0", "q4_0", "q4_k"])
@pytest.mark.parametrize("form", SHAPES)
def test_arbitrary_bytes(ctx, fmt, form):
    # any bytes: block scales may be Inf, NaN or subnormal f16 values
    in_f, (batch, out_f) = length(fmt, 1), SHAPES[form]
    numel, nbytes = vtq.BLOCK[FORMATS[fmt][0]]
    w = O.lcg_bytes(out_f * (in_f // numel) * nbytes, 0xC0DE)
    compare(ctx, fmt, form, synth.activations(batch * in_f, seed=29), w, in_f)


@pytest.mark.parametrize("fmt", ["f32", "q8_0"])
def test_short_rows_on_two_token_tiles(ctx, fmt):
    in_f, (batch, out_f) = {"f32": 161, "q8_0": 96}[fmt], SHAPES[21]
    compare(ctx, fmt, 21, synth.activations(batch * in_f, seed=31), weights(fmt, out_f, in_f, 37), in_f)
