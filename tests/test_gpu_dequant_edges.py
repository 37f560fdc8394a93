"""Dequantization and the embedding gather at the edges of their four-element
split: one block, the last quads of a workgroup's 4096 elements, element
counts that are no multiple of four (F32, F16), rows of an odd length, and
buffers that start at any byte (the blocks) or any float (the output).
Bit-exact against the oracle, as dequantize_f32 (src/gguf/dequant.rs:10-31)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from inferox_amd import _native
from inferox_amd.gguf_writer import F16, F32, Q4_0, Q8_0, Q8_K
from oracle import binding as orc
from tests.gpu_util import Dev, Tensor
from tests.test_gpu_kernels import ALL, BLOCK, _raw, _same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("shift", [0, 1, 2, 5])
def test_raw_stream_edges(t, shift):
    be = BLOCK.get(t, (1, 0))[0]
    rng = np.random.default_rng(900 + t + shift)
    for n in {be, 3 * be, 4096 - be, 4096, 4096 + be, 5 * 4096 + 7 * be}:
        raw = _raw(t, n, rng, special=True)
        src = Dev.of(np.concatenate([np.zeros(shift, np.uint8), raw]))
        out = Dev.of(np.full(n + 16, 7.0, np.float32))
        rc = _native.lib().ifx_dequantize_f32(t, n, C.c_void_p(src.ptr.value + shift), raw.size,
                                              C.c_void_p(out.ptr.value + 4 * shift), n, None)
        assert rc == 0
        got = out.get(np.float32, n + 16)
        _, ref = orc.dequantize(t, raw, n)
        ok, bad = _same_bits(got[shift:shift + n], ref)
        assert ok, f"n {n}: {bad} elements differ"
        assert np.all(got[:shift] == 7.0) and np.all(got[shift + n:] == 7.0), f"n {n}: written outside"


@pytest.mark.parametrize("t,cols", [(F32, 3), (F32, 1028), (F16, 7), (F16, 1030), (Q4_0, 32), (Q8_0, 1056),
                                    (Q8_K, 256)])
def test_rows_and_gather_edges(t, cols):
    rows = 19
    rng = np.random.default_rng(950 + t + cols)
    raw = _raw(t, rows * cols, rng, special=True)
    w = Tensor(t, raw, rows, cols)
    _, ref = orc.dequantize(t, raw, rows * cols)
    ref = np.asarray(ref, np.float32).reshape(rows, cols)
    out = Dev(4 * rows * cols)
    assert _native.lib().ifx_tensor_dequant(w.h, out.ptr, None) == 0
    ok, bad = _same_bits(out.get(np.float32, rows * cols), ref.reshape(-1))
    assert ok, f"{bad} elements differ"
    ids = np.array([18, 0, 7, 7], np.uint32)
    d_ids, g = Dev.of(ids), Dev.of(np.full(4 * cols + 4, 7.0, np.float32))
    assert _native.lib().ifx_ops_embedding_lookup(w.h, d_ids.ptr, 4, C.c_void_p(g.ptr.value + 4), None) == 0
    got = g.get(np.float32, 4 * cols + 4)
    ok, bad = _same_bits(got[1:1 + 4 * cols], ref[ids].reshape(-1))
    assert ok and got[0] == 7.0 and np.all(got[1 + 4 * cols:] == 7.0), f"{bad} elements differ"
