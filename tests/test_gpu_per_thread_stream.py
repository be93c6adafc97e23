"""hipStreamPerThread is one handle for another stream in every thread: batches
on it must not take a workspace by the handle, which two threads would share.
"""
import threading

import pytest

import oracle as O
import vtq
from vtq import synth

from test_gpu_parity import THREADS, assert_bits_equal

pytestmark = pytest.mark.gpu

PER_THREAD = 2  # hipStreamPerThread


def _case(t, batch, in_f, out_f, seed):
    import torch

    w = synth.weights(t, out_f, in_f, seed=seed)
    x = synth.activations(batch * in_f, seed=seed + 1)
    dy = torch.full((batch * out_f,), float("nan"), device="cuda")
    return torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda(), dy, O.linear_dispatch(t, 0, x, w, batch, in_f, out_f, THREADS)


def _call(c, shape, case, stream):
    t, b, i_f, o_f = shape
    dx, dw, dy, _ = case
    c.linear_device(t, 0, dx.data_ptr(), dw.data_ptr(), dw.numel(), dy.data_ptr(), b, i_f, o_f, stream)


@pytest.mark.parametrize("shape", [(vtq.Q6_K, 16, 2048, 900), (vtq.Q4_K, 16, 2048, 900)])
def test_no_workspace_is_made(shape):
    import torch

    case = _case(*shape, seed=3)
    with vtq.Context(0) as warm:  # both forms' code loaded
        _call(warm, shape, case, None)
        _call(warm, shape, case, PER_THREAD)
        torch.cuda.synchronize()
    with vtq.Context(0) as c:
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info(0)[0]
        _call(c, shape, case, PER_THREAD)
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info(0)[0] == free
        assert_bits_equal(case[2].cpu().numpy(), case[3], str(shape))


def test_two_threads_take_turns_on_one_context():
    import torch

    shapes = [(vtq.Q6_K, 40, 4096, 2000), (vtq.Q6_K, 24, 4096, 1500)]
    cases = [_case(*s, seed=20 + i) for i, s in enumerate(shapes)]
    torch.cuda.synchronize()
    turn, errors = threading.Barrier(2, timeout=60), []
    with vtq.Context(0) as c:
        def work(k):
            try:
                for _ in range(4):
                    for who in (0, 1):  # one thread at a time on the context
                        if who == k:
                            _call(c, shapes[k], cases[k], PER_THREAD)
                        turn.wait()
            except Exception as e:  # noqa: BLE001
                errors.append(e)
                turn.abort()

        threads = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
        assert not errors, errors
        for shape, case in zip(shapes, cases):
            assert_bits_equal(case[2].cpu().numpy(), case[3], str(shape))
