"""Workspaces kept between operator calls: calls of growing and shrinking
sizes, from several threads at once, half of them on streams of their own, give
what a lone call gives (bit for bit: the summation order does not depend on the
workspace), also with matrices uploaded after the last one was freed. (That
freeing it gives back what is kept: test_host_memory.py.)"""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

from inferox_amd import _native, synth
from inferox_amd.gguf_writer import Q4_K
from tests.gpu_util import Dev, Tensor
from tests.test_gpu_other_capture import NON_BLOCKING, _hip as hip

pytestmark = pytest.mark.gpu

L = _native.lib
SHAPES = [(2, 512, 256), (70, 1024, 512), (300, 512, 1024), (3, 2048, 512), (513, 256, 256), (3, 512, 4096)]  # the last cuts K


def _linear(case, seed):
    m, rows, cols = case
    w = Tensor(Q4_K, synth.random_centred_blocks(Q4_K, rows * cols, cols, "q", seed), rows, cols)
    a = Dev.of(np.random.default_rng(seed).standard_normal(m * cols).astype(np.float32))
    return w, a


def _run_linear(case, w, a, stream=None):
    m, rows, _ = case
    c = Dev(4 * m * rows)
    assert L().ifx_matmul_qt(a.ptr, m, w.h, c.ptr, stream) == 0
    assert L().ifx_stream_synchronize(stream) == 0
    return c.get(np.float32, m * rows)


def _attn(rows, seed):
    r = np.random.default_rng(seed)
    k, v = (Dev.of(r.standard_normal(2 * (rows + 8) * 64).astype(np.float32)) for _ in range(2))
    return Dev.of(r.standard_normal(8 * 64).astype(np.float32)), k, v


def _run_attn(rows, q, k, v, stream=None):
    out = Dev(4 * 8 * 64)
    assert L().ifx_ops_attention_decode(q.ptr, k.ptr, v.ptr, 0, rows + 8, rows, 8, 2, 64, out.ptr, stream) == 0
    return out.get(np.float32, 8 * 64)


def test_calls_of_all_sizes_and_threads_agree():
    lin = [(c, *_linear(c, 10 + i)) for i, c in enumerate(SHAPES)]
    att = [(n, *_attn(n, 20 + n)) for n in (1, 65, 3000, 130)]
    want_l, want_a = [_run_linear(*x) for x in lin], [_run_attn(*x) for x in att]
    bad = []

    streams = [None] * 6
    for i in (1, 3, 5):
        streams[i] = C.c_void_p()
        assert hip().hipStreamCreateWithFlags(C.byref(streams[i]), NON_BLOCKING) == 0

    def work(i):
        try:
            for k in range(6):
                x = (i + k) % len(lin)
                if not np.array_equal(_run_linear(*lin[x], streams[i]), want_l[x]):
                    bad.append(("linear", SHAPES[x]))
                y = (i + k) % len(att)
                if not np.array_equal(_run_attn(*att[y], streams[i]), want_a[y]):
                    bad.append(("attention", att[y][0]))
        except Exception as e:  # noqa: BLE001 - reported by the assertion below
            bad.append(repr(e))

    th = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for st in streams:
        if st is not None:
            hip().hipStreamDestroy(st)
    assert not bad, bad
    del lin  # the last matrices
    again = _linear(SHAPES[1], 11)
    assert np.array_equal(_run_linear(SHAPES[1], *again), want_l[1])


def test_a_request_past_what_is_kept():
    """64 MiB of operands and more (not kept) between two small calls."""
    small, big = (5, 512, 256), (16384, 256, 4096)
    s, b = _linear(small, 31), _linear(big, 32)
    first = _run_linear(small, *s)
    y = _run_linear(big, *b)
    assert np.array_equal(_run_linear(big, *b), y)
    assert np.array_equal(_run_linear(small, *s), first)
    row = Dev(4 * 256)
    assert L().ifx_gemv(b[0].h, C.c_void_p(b[1].ptr.value + 4 * 4096 * 16383), row.ptr, None) == 0
    one = row.get(np.float32, 256)
    got = y.reshape(16384, 256)[16383]
    assert np.linalg.norm(got - one) <= 4e-6 * np.linalg.norm(one)  # 22-bit operands on both sides


def test_after_an_allocation_that_failed():
    """An allocation no device has room for gives up what is kept and fails; calls
    after it start afresh and give what they gave."""
    lin, att = _linear(SHAPES[1], 41), _attn(3000, 42)
    want = _run_linear(SHAPES[1], *lin), _run_attn(3000, *att)
    p = C.c_void_p()
    assert L().ifx_malloc(C.byref(p), 1 << 42) != 0
    for _ in range(2):
        assert np.array_equal(_run_linear(SHAPES[1], *lin), want[0])
        assert np.array_equal(_run_attn(3000, *att), want[1])
