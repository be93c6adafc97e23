"""GPU parity of the k-quant GEMMs at the batches and formats they take over from
the per-row GEMV: Q6_K from 3 rows, Q4_K from 4 to 31 rows.  Bit for bit
against the oracle; the per-stream workspace slots and graph capture against
the same calls made one at a time.
"""
import numpy as np
import pytest

import oracle as O
import vtq
from vtq import synth

from test_gpu_parity import F, THREADS, assert_bits_equal, check

pytestmark = pytest.mark.gpu

# every tree shape of short rows, piece sizes 1..16 of longer ones, token and
# row counts either side of the 32 x 32 tiles, both sides of the batch rule
Q6K_SHAPES = [(8, 256, 1), (9, 256, 33), (31, 512, 31), (32, 768, 32), (33, 1024, 65), (40, 1280, 130), (64, 2048, 513),
              (65, 3840, 97), (8, 4096, 300), (3, 4096, 2049), (2, 4096, 2049), (7, 4096, 40), (20, 17 * 256, 70),
              (33, 22 * 256, 260), (12, 33 * 256, 129), (70, 43 * 256, 64), (16, 64 * 256, 40), (8, 97 * 256, 33), (9, 71 * 256, 40), (8, 95 * 256, 33),
              (11, 126 * 256, 40), (11, 127 * 256, 40), (9, 128 * 256, 20), (300, 2048, 1500)]
Q4K_SHAPES = [(16, 256, 1), (17, 512, 33), (31, 1024, 70), (8, 4096, 1025), (4, 4096, 8200), (9, 22 * 256, 800),
              (16, 43 * 256, 100), (5, 43 * 256, 2500), (24, 127 * 256, 34), (16, 128 * 256, 9)]


# two token tiles to a wave: one to eight waves, pieces of 4, 8 and 16 leaves, a
# last pair of one tile, remainders of rows and tokens
Q6K_SHAPES += [(65, 512, 12001), (96, 2048, 5700), (70, 15 * 256, 2610), (40, 4096, 5701), (33, 22 * 256, 5200),
               (64, 43 * 256, 5130), (33, 64 * 256, 5130), (33, 72 * 256, 5121), (50, 96 * 256, 5130)]


@pytest.mark.parametrize("batch,in_f,out_f", Q6K_SHAPES)
def test_q6k_batch(ctx, batch, in_f, out_f):
    w = synth.weights(vtq.Q6_K, out_f, in_f, seed=in_f * 3 + out_f)
    check(ctx, vtq.Q6_K, 0, synth.activations(batch * in_f, seed=in_f + batch), w, batch, in_f, out_f)


@pytest.mark.parametrize("batch,in_f,out_f", Q4K_SHAPES)
def test_q4k_small_batch(ctx, batch, in_f, out_f):
    w = synth.weights(vtq.Q4_K, out_f, in_f, seed=in_f * 5 + out_f)
    check(ctx, vtq.Q4_K, 0, synth.activations(batch * in_f, seed=in_f + 3 * batch), w, batch, in_f, out_f)


# batches walked in chunks: 8192 tokens a launch; 8 MiB of workspace (1897
# tokens of 17 super-blocks)
@pytest.mark.parametrize("batch,in_f,out_f", [(8193, 256, 40), (2000, 17 * 256, 33)])
def test_q6k_batch_chunks(ctx, batch, in_f, out_f):
    w = synth.weights(vtq.Q6_K, out_f, in_f, seed=in_f + out_f)
    check(ctx, vtq.Q6_K, 0, synth.activations(batch * in_f, seed=batch), w, batch, in_f, out_f)


@pytest.mark.parametrize("scale", [0x80, 0x7F, 0x81, 0x00, 0xFF, None])
def test_q6k_batch_extreme_scales(ctx, scale):
    # every scale -128, 127, -127, 0, -1 (the two-byte split of code * scale at
    # its ends), or arbitrary block bytes; activations whose codes are all +-127
    batch, in_f, out_f = 40, 1024, 70
    w = O.lcg_bytes(out_f * (in_f // 256) * 210, 0xBEEF).reshape(-1, 210)
    if scale is not None:
        w[:, 192:208] = scale
        w[:, 208:210] = np.frombuffer(np.uint16(0x2E66).tobytes(), np.uint8)
        w[::3, :192] = 0x00  # every code 0: -32
        w[1::3, :192] = 0xFF  # every code 63: 31
    x = synth.activations(batch * in_f, seed=8).reshape(batch, in_f)
    x[0], x[1], x[2], x[3] = 1.0, -1.0, 0.0, -0.0
    x[4, :256], x[5, 7] = np.nan, np.inf
    x[6] = (x[6] * F(1e-42)).astype(F)
    x[7] = (x[7] * F(3e37)).astype(F)
    check(ctx, vtq.Q6_K, 0, x.reshape(-1), w.reshape(-1), batch, in_f, out_f)


def _device_case(t, batch, in_f, out_f, seed):
    import torch

    w = synth.weights(t, out_f, in_f, seed=seed)
    x = synth.activations(batch * in_f, seed=seed + 1)
    want = O.linear_dispatch(t, 0, x, w, batch, in_f, out_f, THREADS)
    dy = torch.full((batch * out_f,), float("nan"), device="cuda")
    return torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), dy, want


def test_batches_on_several_streams():
    # ten streams that do not wait for each other: eight have a workspace of
    # their own, the last two take the forms without one
    import torch

    shapes = [(vtq.Q6_K, 40, 4096, 3000), (vtq.Q4_K, 16, 4096, 3000), (vtq.Q6_K, 64, 2048, 2000), (vtq.Q4_K, 48, 2048, 2000),
              (vtq.Q6_K, 33, 1024, 500), (vtq.Q4_K, 20, 1024, 500), (vtq.Q6_K, 9, 2048, 900), (vtq.Q4_K, 33, 1024, 700),
              (vtq.Q6_K, 20, 2048, 2000), (vtq.Q4_K, 24, 2048, 2000)]
    cases = [_device_case(*s, seed=100 + i) for i, s in enumerate(shapes)]
    with vtq.Context(0) as c:
        # stream handles of this test alone, whatever torch's pool hands out twice
        streams = {s.cuda_stream: s for s in (torch.cuda.Stream() for _ in range(64))}
        streams = list(streams.values())[:len(shapes)]
        assert len(streams) == len(shapes)
        torch.cuda.synchronize()
        for _ in range(3):
            for (t, b, i_f, o_f), (dx, dw, dy, _w), s in zip(shapes, cases, streams):
                c.linear_device(t, 0, dx.data_ptr(), dw.data_ptr(), dw.numel(), dy.data_ptr(), b, i_f, o_f, s.cuda_stream)
        torch.cuda.synchronize()
        for s, (_x, _w, dy, want) in zip(shapes, cases):
            assert_bits_equal(dy.cpu().numpy(), want, str(s))


def test_captured_batches_share_no_workspace():
    # two graphs captured on one stream, replayed side by side on two others
    import torch

    shapes = [(vtq.Q6_K, 40, 4096, 3000), (vtq.Q6_K, 24, 4096, 2500)]
    cases = [_device_case(*s, seed=400 + i) for i, s in enumerate(shapes)]
    with vtq.Context(0) as c:
        cap, graphs = torch.cuda.Stream(), []
        for (t, b, i_f, o_f), (dx, dw, dy, _w) in zip(shapes, cases):
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], stream=cap):
                c.linear_device(t, 0, dx.data_ptr(), dw.data_ptr(), dw.numel(), dy.data_ptr(), b, i_f, o_f, cap.cuda_stream)
        streams = [torch.cuda.Stream() for _ in graphs]
        for _ in range(3):
            for _x, _w, dy, _want in cases:
                dy.fill_(float("nan"))
            torch.cuda.synchronize()
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
            torch.cuda.synchronize()
            for s, (_x, _w, dy, want) in zip(shapes, cases):
                assert_bits_equal(dy.cpu().numpy(), want, str(s))
        del graphs


@pytest.mark.parametrize("t,batch,in_f,out_f", [(vtq.Q6_K, 40, 4096, 700), (vtq.Q4_K, 16, 4096, 700), (vtq.Q8_0, 64, 4096, 700),
                                                (vtq.Q4_K, 40, 4096, 700)])
def test_first_batch_call_under_graph_capture(t, batch, in_f, out_f):
    # a fresh context's first call is captured (without a workspace, or in the
    # slot that captured calls share), then replayed with other inputs between eager calls
    import torch

    dx, dw, dy, want = _device_case(t, batch, in_f, out_f, seed=300)
    x2 = synth.activations(batch * in_f, seed=777)
    want2 = O.linear_dispatch(t, 0, x2, dw.cpu().numpy(), batch, in_f, out_f, THREADS)
    with vtq.Context(0) as c:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            c.linear_device(t, 0, dx.data_ptr(), dw.data_ptr(), dw.numel(), dy.data_ptr(), batch, in_f, out_f,
                            torch.cuda.current_stream().cuda_stream)
        x1 = dx.clone()
        for x, w in ((x1, want), (torch.from_numpy(x2).cuda(), want2), (x1, want)):
            dx.copy_(x)
            dy.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert_bits_equal(dy.cpu().numpy(), w, "replay")
            c.linear_device(t, 0, dx.data_ptr(), dw.data_ptr(), dw.numel(), dy.data_ptr(), batch, in_f, out_f, None)
            torch.cuda.synchronize()
            assert_bits_equal(dy.cpu().numpy(), w, "eager")
        del g
