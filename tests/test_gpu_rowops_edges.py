"""rms_norm_rows, swiglu and add_in_place at the edges of their four-element
forms: lengths around a multiple of four, rows around 1024 quads and 16384
columns, pointers that are not 16-byte aligned, outputs that are an input."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from inferox_amd import _native
from tests.gpu_util import Dev

pytestmark = pytest.mark.gpu


def _at(d, off):
    return C.c_void_p(d.ptr.value + 4 * off)


@pytest.mark.parametrize("n", [1, 4, 64, 257, 288, 4092, 4096, 4100, 16384, 16388])
@pytest.mark.parametrize("off", [0, 1])
def test_rms_norm_rows(n, off):
    r = np.random.default_rng(n + off)
    rows = 3
    x = r.standard_normal((rows, n)).astype(np.float32)
    x[1] *= 1e3
    w = (1 + 0.1 * r.standard_normal(n)).astype(np.float32)
    pad = np.full(off, 7.0, np.float32)
    d = Dev.of(np.concatenate([pad, x.reshape(-1), [7.0]]).astype(np.float32))
    d_w = Dev.of(np.concatenate([pad, w]).astype(np.float32))
    assert _native.lib().ifx_ops_rms_norm_rows(_at(d, off), _at(d_w, off), n, rows, 1e-5, None) == 0
    got = d.get(np.float32, off + rows * n + 1)
    assert np.all(got[:off] == 7.0) and got[-1] == 7.0
    x64 = x.astype(np.float64)
    ref = x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-5) * w
    # a sum of n squares (relative error below 64 roundings: 16 per lane, the
    # rest a tree), a root, a division, two products
    assert np.all(np.abs(got[off:-1].reshape(rows, n) - ref) <= 70 * 2.0 ** -24 * np.abs(ref) + 1e-30)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 4096 * 256 * 4 + 6])
@pytest.mark.parametrize("off", [0, 1, 4])
def test_elementwise(n, off):
    r = np.random.default_rng(n + off)
    a, b = (np.concatenate([np.zeros(off), 5 * r.standard_normal(n), [7.0]]).astype(np.float32) for _ in range(2))
    d_a, d_b, d_o = Dev.of(a), Dev.of(b), Dev.of(np.full(off + n + 1, 7.0, np.float32))
    L = _native.lib()
    assert L.ifx_ops_swiglu(_at(d_a, off), _at(d_b, off), _at(d_o, off), n, None) == 0
    sep = d_o.get(np.float32, off + n + 1)
    g, u = a[off:-1].astype(np.float64), b[off:-1].astype(np.float64)
    ref = g / (1 + np.exp(-np.clip(g, -80, 80))) * u
    assert np.all(np.abs(sep[off:-1] - ref) <= 8 * 2.0 ** -24 * np.abs(ref) + 1e-30)
    assert np.all(sep[:off] == 7.0) and sep[-1] == 7.0
    assert L.ifx_ops_swiglu(_at(d_a, off), _at(d_b, off), _at(d_a, off), n, None) == 0  # over the gate
    assert np.array_equal(d_a.get(np.float32, off + n + 1)[off:-1], sep[off:-1])
    assert L.ifx_ops_add_in_place(_at(d_a, off), _at(d_b, off), n, None) == 0
    assert np.array_equal(d_a.get(np.float32, off + n + 1)[off:-1], sep[off:-1] + b[off:-1])
