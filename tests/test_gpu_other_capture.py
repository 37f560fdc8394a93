"""A session's calls beside a stream that another thread is capturing: each
session records the graph of its first steps that way, and the runtime's
synchronous copies, fills and device-wide waits fail meanwhile and end that
capture. Every call here must succeed, give what it gives otherwise, and leave
the capture valid."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from inferox_amd import _native, synth
from tests.gpu_util import GpuModel

pytestmark = pytest.mark.gpu

NON_BLOCKING, RELAXED = 1, 2


def _hip():
    with open("/proc/self/maps") as f:
        return C.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))


def _calls(g, kv_f16):
    p = synth.token_ids(12, synth.TINY.vocab, seed=77)
    s = g.session(64, kv_f16=kv_f16)
    rc, toks = s.generate(p, 6)
    assert rc == 0
    rc, more = s.decode_greedy(int(toks[-1]), 4)
    assert rc == 0
    last = C.c_uint32()
    assert _native.lib().ifx_session_last_token(s.h, C.byref(last)) == 0
    k, v = s.kv_export(16)
    assert s.kv_import(k, v, 16) == 0
    rc, lg = s.decode_step(3)
    assert rc == 0
    s.close()
    return toks, more, last.value, k, v, lg


@pytest.mark.parametrize("kv_f16", [False, True])
def test_calls_beside_a_capture(tiny_path, kv_f16):
    g = GpuModel(tiny_path)
    want = _calls(g, kv_f16)
    hip, st, graph = _hip(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(st), NON_BLOCKING) == 0
    assert hip.hipStreamBeginCapture(st, RELAXED) == 0
    try:
        got = _calls(g, kv_f16)
    finally:
        ended = hip.hipStreamEndCapture(st, C.byref(graph))
        hip.hipStreamDestroy(st)
    assert ended == 0
    if graph:
        hip.hipGraphDestroy(graph)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
    g.close()
