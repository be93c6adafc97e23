"""ctypes binding of libvtq_probe.so: a measurement helper of bench.py (a
hand-written read-only stream kernel) and the dispatch rules' answers for
tests.  Not part of the quantized-linear boundary."""
from __future__ import annotations

import ctypes
import os

from . import F32, LIB_DIR, Q4_0, Q4_K, Q5_0, Q6_K, Q8_0, REGIME_INTEGER, load_library

_lib = None


def lib() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        load_library()  # torch first, then the HIP libraries: one HIP runtime per process
        path = os.path.join(LIB_DIR, "libvtq_probe.so")
        if not os.path.exists(path):
            raise ImportError(f"{path} is missing (run __graft_entry__.build())")
        L = ctypes.CDLL(path)
        L.vtqp_stream_read.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p,
                                       ctypes.c_void_p]
        L.vtqp_stream_read.restype = ctypes.c_int
        for f in (L.vtqp_canon_form, L.vtqp_kquant_form):
            f.argtypes = [ctypes.c_int] * 4
            f.restype = ctypes.c_int
        _lib = L
    return _lib


def stream_read(ptr: int, nbytes: int, workgroups: int, sink_ptr: int, stream: int) -> None:
    """Launch a read-only stream of `nbytes` (a multiple of 16) at device
    address `ptr` with `workgroups` workgroups of 256 threads on `stream`."""
    rc = lib().vtqp_stream_read(ptr, nbytes, workgroups, sink_ptr, stream)
    if rc != 0:
        raise RuntimeError(f"vtqp_stream_read: hipError {rc}")


GEMV, LDS_OPERAND, PER_WAVE = 0, 1, 2  # besides split-K: 300 + piece, 600 + piece with two token tiles to a wave


def form(ggml_type: int, regime: int, batch: int, in_feat: int, out_feat: int) -> int:
    """The kernel form that a call takes: GEMV (one slice per batch row); for
    integer Q4_K and Q6_K LDS_OPERAND, PER_WAVE or split-K's number; else, for
    the pinned dot over a batch, 10 * token tiles of a wave + waves to a tile."""
    if ggml_type == Q6_K or (ggml_type == Q4_K and regime == REGIME_INTEGER):
        return lib().vtqp_kquant_form(ggml_type, batch, in_feat, out_feat)
    fmt = {Q8_0: 0, Q5_0: 1, Q4_0: 2, F32: 3, Q4_K: 4}[ggml_type]
    return lib().vtqp_canon_form(fmt, batch, in_feat, out_feat)
