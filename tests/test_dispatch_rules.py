"""The dispatch rules (vtq_rules.h), asked on the CPU: which kernel form a call takes."""
import pytest

import vtq
from vtq import probe

INT, FLOAT = vtq.REGIME_INTEGER, vtq.REGIME_FLOAT_FUSED


@pytest.mark.parametrize("args,form", [
    ((vtq.Q8_0, INT, 1, 4096, 4096), probe.GEMV), ((vtq.Q8_0, INT, 16, 4096, 4096), 14),
    ((vtq.Q8_0, INT, 64, 4096, 4096), 12), ((vtq.Q8_0, INT, 128, 4096, 4096), 11),
    ((vtq.Q8_0, INT, 512, 2048, 2048), 21), ((vtq.Q4_K, FLOAT, 77, 2048, 5632), 11),
    ((vtq.Q4_K, INT, 1, 4096, 4096), probe.GEMV), ((vtq.Q4_K, INT, 512, 4096, 14336), probe.PER_WAVE),
    ((vtq.Q4_K, INT, 512, 11008, 4096), probe.LDS_OPERAND), ((vtq.Q4_K, INT, 8, 4096, 11008), 304),
    ((vtq.Q6_K, INT, 1, 4096, 32000), probe.GEMV), ((vtq.Q6_K, INT, 200, 11008, 4096), 608),
    ((vtq.Q6_K, INT, 16, 4096, 4096), 302),
])
def test_a_shape_of_each_form(args, form):
    assert probe.form(*args) == form
