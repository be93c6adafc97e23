"""vtq_linear_device_noalloc on the batches that have a form without a workspace
(Q6_K, Q4_K below 32 rows, the pinned dot): they leave the per-GPU array alone,
so they may overlap on streams and contexts.  Bit for bit against the oracle.
"""
import ctypes

import numpy as np
import pytest

import oracle as O
import vtq
from vtq import synth

from test_gpu_parity import THREADS, assert_bits_equal
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu

# (type, batch, in, out): batches that the allocating entry point gives to the GEMM
CASES = [(vtq.Q6_K, 9, 2048, 700), (vtq.Q6_K, 40, 4096, 1500), (vtq.Q4_K, 8, 4096, 1100), (vtq.Q4_K, 31, 1024, 900)]


def _case(t, batch, in_f, out_f, seed):
    import torch

    w = synth.weights(t, out_f, in_f, seed=seed)
    x = synth.activations(batch * in_f, seed=seed + 1)
    dy = torch.full((batch * out_f,), float("nan"), device="cuda")
    return torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), dy, O.linear_dispatch(t, 0, x, w, batch, in_f, out_f, THREADS)


def _call(c, case, shape, stream):
    t, b, i_f, o_f = shape
    dx, dw, dy, _ = case
    rc = _noalloc(c)(c.handle, t, 0, dx.data_ptr(), dw.data_ptr(), dw.numel(), dy.data_ptr(), b, i_f, o_f, stream)
    assert rc == 0, c.lib.vtq_last_error(c.handle)


def _hip():
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
    return ctypes.CDLL(path)


def _launches(c, case, shape):
    """Kernels that the call launches: the nodes of its capture, which is never run."""
    import torch

    hip, s = _hip(), torch.cuda.Stream()
    graph, n = ctypes.c_void_p(), ctypes.c_size_t()
    hip.hipStreamBeginCapture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    hip.hipStreamEndCapture.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    hip.hipGraphGetNodes.argtypes = [ctypes.c_void_p] * 3
    hip.hipGraphDestroy.argtypes = [ctypes.c_void_p]
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(s.cuda_stream, 2) == 0
    try:
        _call(c, case, shape, s.cuda_stream)
    finally:
        assert hip.hipStreamEndCapture(s.cuda_stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    return n.value


@pytest.mark.parametrize("shape", CASES)
def test_one_launch_and_no_pre_pass(shape):
    # a GEMM is two launches, the first of which fills the workspace
    with vtq.Context(0) as c:
        assert _launches(c, _case(*shape, seed=11), shape) == 1


def test_a_gemm_call_is_two_launches():
    shape = (vtq.Q4_K, 40, 1024, 300)
    with vtq.Context(0) as c:
        assert _launches(c, _case(*shape, seed=13), shape) == 2


@pytest.mark.parametrize("contexts", [1, 2])
def test_calls_overlap_on_streams_and_contexts(contexts):
    import torch

    cases = [_case(*s, seed=50 + i) for i, s in enumerate(CASES)]
    cs = [vtq.Context(0) for _ in range(contexts)]
    try:
        streams = [torch.cuda.Stream() for _ in CASES]
        torch.cuda.synchronize()
        for _ in range(5):
            for i, (shape, case, s) in enumerate(zip(CASES, cases, streams)):
                _call(cs[i % contexts], case, shape, s.cuda_stream)
        torch.cuda.synchronize()
        for shape, case in zip(CASES, cases):
            assert_bits_equal(case[2].cpu().numpy(), case[3], str(shape))
    finally:
        for c in cs:
            c.close()


def test_graphs_replayed_side_by_side():
    import torch

    shapes = CASES[1:3]
    cases = [_case(*s, seed=80 + i) for i, s in enumerate(shapes)]
    with vtq.Context(0) as c:
        graphs = []
        for shape, case in zip(shapes, cases):
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1]):
                _call(c, case, shape, torch.cuda.current_stream().cuda_stream)
        streams = [torch.cuda.Stream() for _ in graphs]
        for _ in range(3):
            for case in cases:
                case[2].fill_(float("nan"))
            torch.cuda.synchronize()
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
            torch.cuda.synchronize()
            for shape, case in zip(shapes, cases):
                assert_bits_equal(case[2].cpu().numpy(), case[3], str(shape))
        del graphs
