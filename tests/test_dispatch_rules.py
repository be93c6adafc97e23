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


@pytest.mark.parametrize("in_f,out_f", [(17 * 256, 8200), (5120, 60000), (8192, 128256), (11008, 16384), (14336, 8192),
                                        (16384, 9000), (28672, 8192), (127 * 256, 20000), (43 * 256, 4096)])
@pytest.mark.parametrize("batch", [4, 5, 8, 16, 31])
def test_q4k_batches_below_32_on_long_rows_take_split_k(batch, in_f, out_f):
    # never the LDS-operand kernel, a workgroup of which holds 128 tokens: slower than the GEMV at 4 and 5 rows
    assert probe.form(vtq.Q4_K, INT, batch, in_f, out_f) >= 300


@pytest.mark.parametrize("in_f", [2048, 3072, 4096])
def test_four_q4k_rows_past_the_split_k_grids(in_f):
    assert [probe.form(vtq.Q4_K, INT, 4, in_f, n) for n in (32769, 39999)] == [probe.GEMV] * 2
    assert [probe.form(vtq.Q4_K, INT, 4, in_f, n) for n in (40000, 65536)] == [probe.PER_WAVE] * 2
    assert probe.form(vtq.Q4_K, INT, 5, in_f, 32769) == probe.PER_WAVE
    assert probe.form(vtq.Q4_K, INT, 4, in_f, 32768) >= 300


@pytest.mark.parametrize("batch,in_f,below,above", [(3, 1024, 8191, 8192), (3, 2048, 5119, 5120), (3, 4096, 4095, 4096),
                                                    (3, 8192, 4095, 4096), (3, 14336, 2340, 2341), (4, 4096, 2047, 2048),
                                                    (4, 8192, 2047, 2048), (4, 14336, 804, 805), (5, 8192, 1407, 1408),
                                                    (5, 14336, 585, 586), (7, 8192, 1023, 1024)])
def test_q6k_small_batches_of_long_rows(batch, in_f, below, above):
    # the GEMV is faster below: 3 rows of 14336 -> 600 18.6 us against 25.3
    assert probe.form(vtq.Q6_K, INT, batch, in_f, below) == probe.GEMV
    assert probe.form(vtq.Q6_K, INT, batch, in_f, above) > probe.GEMV


@pytest.mark.parametrize("in_f", [256, 4096, 126 * 256])
def test_q6k_batches_of_eight_rows_take_the_gemm(in_f):
    assert probe.form(vtq.Q6_K, INT, 2, in_f, 100000) == probe.GEMV
    assert probe.form(vtq.Q6_K, INT, 8, in_f, 1) >= 300
    assert probe.form(vtq.Q6_K, INT, 8, 127 * 256, 1) == probe.GEMV


@pytest.mark.parametrize("t,in_f,out_f", [(vtq.Q4_0, 1536, 32000), (vtq.Q4_0, 3072, 16384), (vtq.Q4_0, 4096, 16384),
                                          (vtq.Q4_0, 8192, 32000), (vtq.Q8_0, 4352, 32000), (vtq.Q8_0, 8192, 32000)])
def test_two_rows_on_a_full_grid_stay_with_the_gemv(t, in_f, out_f):
    # Q4_0 2 x 4096 -> 16384 47.5 us against 57.0 in the batch kernel; three rows 67.5 against 56.9
    assert probe.form(t, INT, 2, in_f, out_f) == probe.GEMV
    assert probe.form(t, INT, 3, in_f, out_f) > probe.GEMV


@pytest.mark.parametrize("t,in_f,out_f", [(vtq.Q4_0, 11008, 16384), (vtq.Q8_0, 14336, 32000), (vtq.Q5_0, 4096, 14336),
                                          (vtq.F32, 4096, 14336)])
def test_two_rows_that_take_the_batch_kernel(t, in_f, out_f):
    assert probe.form(t, INT, 2, in_f, out_f) > probe.GEMV
