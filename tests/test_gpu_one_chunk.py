"""Decode attention whose rows fit one 64-row chunk writes its output without a
merge: the operator over 1, 63, 64 (one chunk) and 65 rows (two, merged)
against float64, and a session's steps across the 64-row line giving the bits
of the separate-merge steps (fixed summation order, the merge forced)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from inferox_amd import _native, synth
from tests.gpu_util import Dev, GpuModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("heads,kv_heads,hd", [(6, 6, 48), (8, 2, 128), (16, 2, 128), (8, 2, 64), (6, 2, 96), (4, 4, 128)])
def test_rows_around_one_chunk(heads, kv_heads, hd, f16):
    r = np.random.default_rng(heads + hd)
    seq, dt = 80, np.float16 if f16 else np.float32
    q = r.standard_normal((heads, hd)).astype(np.float32)
    k, v = (r.standard_normal((kv_heads, seq, hd)).astype(dt) for _ in range(2))
    d_q, d_k, d_v = Dev.of(q), Dev.of(k), Dev.of(v)
    for rows in (1, 2, 63, 64, 65):
        out = Dev(4 * heads * hd)
        assert _native.lib().ifx_ops_attention_decode(d_q.ptr, d_k.ptr, d_v.ptr, int(f16), seq, rows, heads, kv_heads,
                                                      hd, out.ptr, None) == 0
        got = out.get(np.float32, heads * hd).reshape(heads, hd)
        for h in range(heads):
            kk, vv = (x[h * kv_heads // heads, :rows].astype(np.float64) for x in (k, v))
            s = kk @ q[h].astype(np.float64) / np.sqrt(hd)
            e = np.exp(s - s.max())
            ref = (e / e.sum()) @ vv
            # scores: hd f32 products and sums (|s| to ~10): 2e-5 of each weight at most
            assert np.abs(got[h] - ref).max() <= 4e-5 * np.abs(vv).max(), (rows, h)


@pytest.mark.parametrize("rows", [40, 64, 65])
@pytest.mark.parametrize("where", ["q", "q+1", "q-1", "k", "v"])
def test_output_over_the_inputs(rows, where):
    """The output may overwrite what the attention reads: q itself, q a head
    further on or back, rows of a cache. Bit for bit what lies apart gives."""
    heads, kv_heads, hd, seq = 32, 8, 128, 80
    r = np.random.default_rng(rows)
    q = r.standard_normal(heads * hd).astype(np.float32)
    k, v = (r.standard_normal(kv_heads * seq * hd).astype(np.float32) for _ in range(2))
    buf = np.concatenate([np.zeros(hd, np.float32), q, np.zeros(hd, np.float32)])

    def run(over):
        d_q, d_k, d_v, d_o = Dev.of(buf), Dev.of(k), Dev.of(v), Dev(4 * heads * hd)
        at = {"": (d_o, 0), "q": (d_q, hd), "q+1": (d_q, 2 * hd), "q-1": (d_q, 0), "k": (d_k, 3 * seq * hd),
              "v": (d_v, 2 * seq * hd)}[over]
        ptr = C.c_void_p(at[0].ptr.value + 4 * at[1])
        assert _native.lib().ifx_ops_attention_decode(C.c_void_p(d_q.ptr.value + 4 * hd), d_k.ptr, d_v.ptr, 0, seq, rows,
                                                      heads, kv_heads, hd, ptr, None) == 0
        return at[0].get(np.float32, at[0].nbytes // 4)[at[1]:at[1] + heads * hd]

    assert np.array_equal(run(where), run(""))


def test_steps_across_the_line(tiny_path, monkeypatch):
    g = GpuModel(tiny_path)
    ids = synth.token_ids(70, g.vocab, seed=5)

    def steps():
        s = g.session(96)
        s.set_deterministic(True)
        out = [s.decode_step(int(t))[1] for t in ids]
        s.close()
        return np.array(out)

    def separate(monkeypatch):  # not deterministic: the merge forced into its own launch
        monkeypatch.setenv("IFX_MERGE_O", "0")
        s = g.session(96)
        out = [s.decode_step(int(t))[1] for t in ids]
        s.close()
        monkeypatch.delenv("IFX_MERGE_O")
        return np.array(out)

    # Q8_0 launches have one summation order, deterministic session or not
    assert np.array_equal(steps(), separate(monkeypatch))
    g.close()
