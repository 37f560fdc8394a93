"""matmul_qt of 2 to 64 rows (the launch that takes a few tokens) at the edges
of its token tiles (16, 32, 64 rows), row tiles (16, 64 .. 256 weight rows) and
256-column blocks: short last blocks (Q8_0, Q4_0), K cut over workgroups or
not, rows of very different magnitude, zero rows, ggml's Q6_K, an output that
overlaps the input, and the m = 65 hand-over to the tile GEMM.

The check is against float64.  The operands carry 22 bits or more (2^-21
relative per product at most, and 2^-38 of the largest activation of its
256-column block, whose scale it shares), the sums are f32: each of the K / 16
matrix instructions and the few scale steps of an output rounds once (2^-24 of
a partial sum, at most sum |a| |w|)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from inferox_amd import _native, synth
from inferox_amd.gguf_writer import Q4_0, Q4_K, Q6_K, Q8_0
from oracle import binding as orc
from tests.gpu_util import Dev, Tensor
from tests.test_gpu_kernels import _raw

pytestmark = pytest.mark.gpu


def _bound(a, w):
    k = a.shape[1]
    b = (2.0 ** -21 + (k / 16 + 16) * 2.0 ** -24) * (np.abs(a) @ np.abs(w).T) + 1e-30
    for c in range(0, k, 256):
        b += 2.0 ** -38 * np.outer(np.abs(a[:, c:c + 256]).max(axis=1), np.abs(w[:, c:c + 256]).sum(axis=1))
    return b


def _weights(t, rows, cols, seed):
    raw = _raw(t, rows * cols, np.random.default_rng(seed))
    _, wf = orc.dequantize(t, raw, rows * cols)
    return Tensor(t, raw, rows, cols), np.asarray(wf, np.float64).reshape(rows, cols)


def _run(w, a, rows, fn="ifx_matmul_qt"):
    m = a.shape[0]
    d_a, d_c = Dev.of(a), Dev.of(np.full(m * rows + 8, 7.0, np.float32))
    assert getattr(_native.lib(), fn)(d_a.ptr, m, w.h, d_c.ptr, None) == 0
    got = d_c.get(np.float32, m * rows + 8)
    assert np.all(got[m * rows:] == 7.0)
    return got[:m * rows].reshape(m, rows).astype(np.float64)


def _check(w, wf, a):
    got = _run(w, a, wf.shape[0])
    ref = a.astype(np.float64) @ wf.T
    over = np.abs(got - ref) / _bound(a.astype(np.float64), wf)
    assert over.max() <= 1.0, f"{over.max():.2f} of the bound at {np.unravel_index(over.argmax(), over.shape)}"


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0, Q4_0])
@pytest.mark.parametrize("rows,cols", [(1, 256), (16, 512), (63, 768), (257, 2560), (1000, 4096)])
def test_tiles_and_tokens(t, rows, cols):
    w, wf = _weights(t, rows, cols, 7 * rows + t)
    for m in (2, 15, 16, 17, 32, 33, 49, 64, 65):
        _check(w, wf, np.random.default_rng(m).standard_normal((m, cols)).astype(np.float32))


@pytest.mark.parametrize("t", [Q8_0, Q4_0])
@pytest.mark.parametrize("rows,cols", [(1, 32), (5, 96), (33, 288), (130, 1056), (64, 4064)])
def test_rows_of_part_blocks(t, rows, cols):
    w, wf = _weights(t, rows, cols, rows + cols + t)
    for m in (2, 16, 31, 64):
        _check(w, wf, np.random.default_rng(m).standard_normal((m, cols)).astype(np.float32))


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
def test_magnitudes(t):
    rows, cols, m = 100, 1024, 20
    w, wf = _weights(t, rows, cols, 31 + t)
    r = np.random.default_rng(5)
    a = r.standard_normal((m, cols))
    a *= 10.0 ** np.linspace(-25, 25, m)[:, None]  # the rows' sizes
    a[3] = 0.0
    a[7, 256:512] = 0.0
    a[8, :256] *= 1e-12  # one block far below its row
    a[9, 700] = 3e30
    _check(w, wf, a.astype(np.float32))


def test_ggml_q6k_scales():
    """int8 scale bytes (ggml's block layout), negative ones among them."""
    rows, cols, m = 48, 512, 18
    r = np.random.default_rng(9)
    raw = r.integers(0, 256, size=(rows * cols // 256, 210), dtype=np.uint8)
    raw[:, 208:210] = r.uniform(1e-4, 1e-2, (raw.shape[0], 1)).astype("<f2").view(np.uint8).reshape(-1, 2)
    h = C.c_void_p()
    flat = np.ascontiguousarray(raw.reshape(-1))
    assert _native.lib().ifx_tensor_upload_ex(Q6_K, flat.ctypes.data_as(C.c_void_p), flat.size, rows, cols, 1,
                                              C.byref(h)) == 0
    w = Tensor.__new__(Tensor)
    w.h, w.rows, w.cols = h, rows, cols
    out = Dev(4 * rows * cols)
    assert _native.lib().ifx_tensor_dequant(w.h, out.ptr, None) == 0
    wf = out.get(np.float32, rows * cols).astype(np.float64).reshape(rows, cols)
    assert (wf < 0).any() and (wf > 0).any()
    _check(w, wf, r.standard_normal((m, cols)).astype(np.float32))


def test_output_over_the_input():
    """C may overwrite A (a square matrix applied in place)."""
    n, m = 512, 9
    raw = synth.random_centred_blocks(Q4_K, n * n, n, "q", 3)
    w = Tensor(Q4_K, raw, n, n)
    _, wf = orc.dequantize(Q4_K, raw, n * n)
    wf = np.asarray(wf, np.float64).reshape(n, n)
    a = np.random.default_rng(4).standard_normal((m, n)).astype(np.float32)
    d = Dev.of(a)
    assert _native.lib().ifx_matmul_qt(d.ptr, m, w.h, d.ptr, None) == 0
    got = d.get(np.float32, m * n).reshape(m, n).astype(np.float64)
    assert np.all(np.abs(got - a.astype(np.float64) @ wf.T) <= _bound(a.astype(np.float64), wf))


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("rows,cols", [(1024, 512), (1024, 2048)])
def test_error_is_no_larger_than_the_tile_gemm(t, rows, cols):
    """Against float64, on activations with a few large channels. The same call
    with its output over its input takes the tile GEMM."""
    few = tile = 0.0
    for seed in range(3):
        raw = synth.random_centred_blocks(t, rows * cols, cols, "q", 50 + seed)
        _, wf = orc.dequantize(t, raw, rows * cols)
        w, wf = Tensor(t, raw, rows, cols), np.asarray(wf, np.float64).reshape(rows, cols)
        for m in (3, 8, 16, 24, 40, 64):
            a = np.random.default_rng(100 * seed + m).standard_normal((m, cols)).astype(np.float32)
            a[:, ::97] *= 8.0
            ref = a.astype(np.float64) @ wf.T
            d = Dev.of(np.concatenate([a.reshape(-1), np.zeros(m * rows, np.float32)]))
            assert _native.lib().ifx_matmul_qt(d.ptr, m, w.h, d.ptr, None) == 0
            over = d.get(np.float32, m * rows).reshape(m, rows)
            n2 = np.sum(ref * ref)
            few += np.sum((_run(w, a, rows) - ref) ** 2) / n2
            tile += np.sum((over - ref) ** 2) / n2
    assert few <= tile, np.sqrt(few / tile)


def test_both_entry_points():
    w, wf = _weights(Q4_K, 640, 2048, 77)
    for m in (3, 40):
        a = np.random.default_rng(m).standard_normal((m, 2048)).astype(np.float32)
        assert np.array_equal(_run(w, a, 640), _run(w, a, 640, "ifx_matmul_qt_noalloc"))
