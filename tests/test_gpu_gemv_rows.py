"""The f32-dot GEMV at the edges of its row split: rows of fewer 16-byte pieces
than lanes (16, 32 or 64 lanes per row), of one to many pieces per lane, of two
to eight waves, odd row counts (the last unit holds one row), and the norm and
RoPE epilogue over each of them.

Against float64.  A lane sums at most 64 products in sequence, then about 16
adds join lanes, waves and scales: 100 roundings of 2^-24 of at most
sum |x| max |w| (twice that for Q8_0 and Q4_0, which sum unsigned quants and
take the offset off)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from inferox_amd import _native
from inferox_amd.gguf_writer import F16, F32, Q4_0, Q8_0, Q8_K
from oracle import binding as orc
from tests.gpu_util import Dev, Tensor
from tests.test_gpu_kernels import _raw

pytestmark = pytest.mark.gpu

COLS = [32, 256, 288, 512, 544, 1024, 1056, 2048, 2080, 4096, 4128, 8192, 8224, 16384, 16416, 32320]


def _weights(t, rows, cols, seed):
    raw = _raw(t, rows * cols, np.random.default_rng(seed))
    _, wf = orc.dequantize(t, raw, rows * cols)
    return Tensor(t, raw, rows, cols), np.asarray(wf, np.float64).reshape(rows, cols)


def _bound(x, wf):
    return 200 * 2.0 ** -24 * np.abs(x).sum() * np.abs(wf).max(axis=1) + 1e-30


@pytest.mark.parametrize("t", [Q8_0, Q4_0, Q8_K, F16, F32])
@pytest.mark.parametrize("cols", COLS)
def test_row_lengths(t, cols):
    if t == Q8_K and cols % 256:
        pytest.skip("Q8_K rows are whole 256-blocks")
    for rows in (1, 2, 7, 130):
        w, wf = _weights(t, rows, cols, rows + cols + t)
        x = np.random.default_rng(cols).standard_normal(cols).astype(np.float32)
        d_x, d_y = Dev.of(x), Dev.of(np.full(rows + 4, 7.0, np.float32))
        assert _native.lib().ifx_gemv(w.h, d_x.ptr, d_y.ptr, None) == 0
        y = d_y.get(np.float32, rows + 4)
        assert np.all(y[rows:] == 7.0)
        err = np.abs(y[:rows] - wf @ x.astype(np.float64))
        assert np.all(err <= _bound(x, wf)), (rows, (err / _bound(x, wf)).max())


@pytest.mark.parametrize("t", [Q8_0, Q4_0, F16, F32])
@pytest.mark.parametrize("rows,cols", [(40001, 288), (9001, 2048), (9001, 4096), (5001, 8192), (2501, 16384),
                                       (1301, 32320)])
def test_rows_past_the_grid(t, rows, cols):
    """More rows than the launch's waves take at once (2048 waves of one to four
    units of two rows, or groups of 2, 4 and 8 waves per unit): each runs three
    units and more, the last round a part of them and the last unit one row."""
    w, wf = _weights(t, rows, cols, rows + t)
    x = np.random.default_rng(rows).standard_normal(cols).astype(np.float32)
    d_x, d_y = Dev.of(x), Dev.of(np.full(rows + 4, 7.0, np.float32))
    for _ in range(2):
        assert _native.lib().ifx_gemv(w.h, d_x.ptr, d_y.ptr, None) == 0
        y = d_y.get(np.float32, rows + 4)
        assert np.all(y[rows:] == 7.0)
        err = np.abs(y[:rows] - wf @ x.astype(np.float64))
        assert np.all(err <= _bound(x, wf)), (np.nonzero(err > _bound(x, wf))[0][:8], (err / _bound(x, wf)).max())


@pytest.mark.parametrize("t", [Q8_0, Q4_0, F16])
@pytest.mark.parametrize("cols", [96, 288, 1056, 4096, 4128, 16416])
def test_norm_and_rope(t, cols):
    """q/k/v of one token (ifx_ops_qkv, the tiled launch), float64 norm and RoPE."""
    hd, nq, nkv, pos, row, seq, eps, base = 16, 48, 16, 5, 3, 8, 1e-5, 10000.0
    mats = [_weights(t, r, cols, cols + i) for i, r in enumerate((nq, nkv, nkv))]
    r = np.random.default_rng(cols)
    x = (3.0 * r.standard_normal(cols)).astype(np.float32)
    nw = (1.0 + 0.1 * r.standard_normal(cols)).astype(np.float32)
    d_x, d_n, d_q = Dev.of(x), Dev.of(nw), Dev(4 * nq)
    d_k, d_v = (Dev.of(np.zeros(nkv * seq, np.float32)) for _ in range(2))
    path = C.c_int()
    assert _native.lib().ifx_ops_qkv(mats[0][0].h, mats[1][0].h, mats[2][0].h, d_x.ptr, d_n.ptr, eps, hd, hd, base,
                                     pos, d_q.ptr, d_k.ptr, d_v.ptr, 0, seq, row, 0, C.byref(path), None) == 0
    x64 = x.astype(np.float64)
    y = x64 / np.sqrt((x64 * x64).mean() + eps) * nw
    inv = (np.float32(1) / np.power(np.float32(base), np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)))
    ang = (np.float32(pos) * inv.astype(np.float32)).astype(np.float64)

    def rope(v):
        v = v.reshape(-1, hd)
        out = np.empty_like(v)
        out[:, 0::2] = v[:, 0::2] * np.cos(ang) - v[:, 1::2] * np.sin(ang)
        out[:, 1::2] = v[:, 0::2] * np.sin(ang) + v[:, 1::2] * np.cos(ang)
        return out.reshape(-1)

    got = [d_q.get(np.float32, nq)]
    for d in (d_k, d_v):  # [kv head][seq][hd]
        got.append(d.get(np.float32, nkv * seq).reshape(nkv // hd, seq, hd)[:, row].reshape(-1))
    for i, (_, wf) in enumerate(mats):
        ref = wf @ y
        # RoPE mixes two rows; the norm scale and the rotation add a few roundings
        bound = np.repeat(_bound(y, wf).reshape(-1, 2).sum(axis=1), 2) * 1.1
        ref = rope(ref) if i < 2 else ref
        assert np.all(np.abs(got[i] - ref) <= bound), i
