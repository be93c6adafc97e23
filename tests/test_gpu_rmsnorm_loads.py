"""RMSNorm rows held in registers (rms_norm_kernel, rows of 1024 to 4096 inputs) against the CPU oracle, bit for bit:
pointers aligned to 4 bytes only, the result written over the input, nothing written past the row."""
import numpy as np
import pytest
import torch

import oracle
from vtq import runtime

from test_gpu_rmsnorm import same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1024, 1088, 2048, 4032, 4096])
@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("inplace", [False, True])
def test_rms_norm_any_alignment(n, shift, inplace):
    rng = np.random.default_rng(n + shift)
    x = rng.standard_normal(n).astype(np.float32)
    w = rng.standard_normal(n).astype(np.float32)
    bx, bw, by = (torch.full((n + 8,), 7.0, device="cuda:0") for _ in range(3))
    bx[shift:shift + n] = torch.from_numpy(x).to("cuda:0")
    bw[shift:shift + n] = torch.from_numpy(w).to("cuda:0")
    out = bx if inplace else by
    runtime.rms_norm_device(bx[shift:].data_ptr(), bw[shift:].data_ptr(), n, np.float32(1e-5), out[shift:].data_ptr(), None)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert same(got[shift:shift + n], oracle.rms_norm(x, w, np.float32(1e-5)))
    assert np.all(got[:shift] == 7.0) and np.all(got[shift + n:] == 7.0)
