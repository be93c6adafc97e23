"""GPU parity of the batched pinned dot (canon_gemm.hip,
canon_gemm_split.hip) against the oracle, bit for bit.

The shapes are large enough for the dispatch to prefer a batch kernel, most of
them its form for small grids (four waves to a tile of 16 rows x 16 tokens), and
have token and row counts either side of the tiles, rows that end in the middle
of a 64-input step, and rows of two and three 8192-input chunks.
test_gpu_canon_forms.py takes every form and format through such rows by name.
"""
import numpy as np
import pytest

import oracle as O
import vtq
from vtq import synth

from test_gpu_parity import F, check

pytestmark = pytest.mark.gpu

BLOCK_SHAPES = [(150, 992, 300), (45, 512, 2011), (300, 64, 9000), (67, 160, 10001), (100, 8224, 240), (90, 16640, 270),
                (150, 1056, 1530)]
Q4K_SHAPES = [(45, 512, 2011), (40, 256, 5000), (260, 256, 9001), (33, 4352, 1030), (34, 8448, 1030), (150, 1280, 1530)]
F32_SHAPES = [(70, 1001, 700), (35, 100, 9003), (260, 33, 9001), (64, 32, 12000), (80, 4097, 513), (65, 8197, 259),
              (150, 1030, 1530)]
CASES = [(t, 0, *s) for t in (vtq.Q8_0, vtq.Q5_0, vtq.Q4_0) for s in BLOCK_SHAPES] \
    + [(vtq.Q4_0, 0, 17, 8288, 6200)] + [(vtq.Q4_K, 1, *s) for s in Q4K_SHAPES] + [(vtq.F32, 0, *s) for s in F32_SHAPES]


def weights(t, out_f, in_f, seed):
    return synth.weights(t, out_f, in_f, seed, sigma=1.0) if t == vtq.F32 else synth.weights(t, out_f, in_f, seed)


@pytest.mark.parametrize("t,regime,batch,in_f,out_f", CASES)
def test_batched_dot(ctx, t, regime, batch, in_f, out_f):
    x = synth.activations(batch * in_f, seed=in_f + 7 * batch)
    check(ctx, t, regime, x, weights(t, out_f, in_f, in_f * 3 + out_f), batch, in_f, out_f)


@pytest.mark.parametrize("t,regime,in_f", [(vtq.Q8_0, 0, 992), (vtq.Q5_0, 0, 992), (vtq.Q4_0, 0, 992),
                                           (vtq.Q4_K, 1, 1024), (vtq.F32, 0, 1001)])
def test_batched_dot_edge_values(ctx, t, regime, in_f):
    # tokens of zeros, of one NaN or infinity at a row's first and last input
    # (the neighbouring tokens must not see them), of products in and below the
    # subnormal range, of sums that overflow
    batch, out_f = 150, 300
    x = synth.activations(batch * in_f, seed=17).reshape(batch, in_f)
    x[0], x[1] = 0.0, -0.0
    x[3, 0], x[5, -1], x[7, 0], x[9, -1] = np.nan, np.nan, np.inf, -np.inf
    x[10:20] *= F(1e-38)
    x[20:30] = (x[20:30] * F(1e-38) * F(1e-6)).astype(F)
    x[30:40] *= F(3e37)
    check(ctx, t, regime, x.reshape(-1), weights(t, out_f, in_f, 23), batch, in_f, out_f)


@pytest.mark.parametrize("t,regime,in_f", [(vtq.Q8_0, 0, 992), (vtq.Q5_0, 0, 992), (vtq.Q4_0, 0, 992),
                                           (vtq.Q4_K, 1, 1024)])
def test_batched_dot_arbitrary_bytes(ctx, t, regime, in_f):
    # any bytes: block scales may be Inf, NaN or subnormal f16 values
    batch, out_f = 150, 300
    numel, nbytes = vtq.BLOCK[t]
    w = O.lcg_bytes(out_f * (in_f // numel) * nbytes, 0xC0DE)
    check(ctx, t, regime, synth.activations(batch * in_f, seed=29), w, batch, in_f, out_f)
