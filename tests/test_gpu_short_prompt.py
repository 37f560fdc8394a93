"""Chunks of up to 64 ids layer by layer, at the edges of the few-row launches'
token tiles (8 rows, 16, 32, 64) and of the rule that chooses them (up to 32
ids, or 64 of a narrow model), against the oracle and against the same ids fed
one at a time (a session whose minimum is 0)."""
from __future__ import annotations

import numpy as np
import pytest

from inferox_amd import synth
from inferox_amd.gguf_writer import Q4_0, Q4_K, Q6_K
from oracle import binding as orc
from tests.conftest import rel_l2
from tests.gpu_util import GpuModel
from tests.test_gpu_prefill import TOL

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tiny(tiny_path):
    g, o = GpuModel(tiny_path), orc.Model(tiny_path)
    yield g, o
    g.close()
    o.close()


@pytest.fixture(scope="module")
def wide(tmpdir_session):
    """Q4_K and Q6_K at the Llama-3-8B width: q/k of one type, v of the other."""
    spec = synth.reduced(synth.LLAMA3_8B, n_layers=2, ctx=512)
    p = str(tmpdir_session / "l8b_2l_short.gguf")
    synth.write_llama(p, spec, seed=8)
    g = GpuModel(p)
    yield g, spec
    g.close()


def _same_rows(got, want, tol=TOL, kv_tol=1e-4):
    (lg, k, v), (lr, kr, vr) = got, want
    assert max(rel_l2(a, b) for a, b in zip(lg, lr)) < tol
    assert rel_l2(k, kr) < kv_tol and rel_l2(v, vr) < kv_tol


def _fed(s, chunks):
    lgs = []
    for ids in chunks:
        rc, lg = s.prefill(ids)
        assert rc == 0
        lgs.append(lg.copy())
    return (np.concatenate(lgs), *s.kv_export(len(s)))


@pytest.mark.parametrize("n", [1, 2, 3, 8, 9, 16, 17, 32, 33, 63, 64])
def test_tiny(tiny, n):
    g, o = tiny
    s, kv = g.session(128), o.kv(128)
    s.set_prefill_batch(1)
    ids = synth.token_ids(n, synth.TINY.vocab, seed=n)
    got = _fed(s, [ids])
    rc, ref = o.prefill(kv, ids)
    assert rc == 0
    _same_rows(got, (ref, *kv.export(n)))
    tok = orc.argmax(ref[-1])[1]
    for _ in range(4):  # decode goes on from the state the chunk left
        rc, lg = s.decode_step(tok)
        _, r = o.decode_step(kv, tok)
        assert rc == 0 and rel_l2(lg, r) < TOL
        tok = orc.argmax(r)[1]
    s.close()


@pytest.mark.parametrize("kv_f16", [False, True])
def test_chunks_of_every_kind(wide, kv_f16):
    """Short chunks, two through the tile GEMMs, then short ones again: the
    workspace grows and is shared. An f16 cache rounds each stored value, so each
    may differ by one of its steps (2^-10 of it at most), and the logits by what
    that does to the attention's scores and sums."""
    g, spec = wide
    ids = synth.token_ids(3 + 32 + 33 + 70 + 9 + 1, spec.vocab, seed=3)
    cuts = np.cumsum([3, 32, 33, 70, 9])
    a, b = g.session(256, kv_f16=kv_f16), g.session(256, kv_f16=kv_f16)
    b.set_prefill_batch(0)
    tols = (2.0 ** -8, 2.0 ** -10) if kv_f16 else (TOL, 1e-4)
    _same_rows(_fed(a, np.split(ids, cuts)), _fed(b, np.split(ids, cuts)), *tols)
    a.close(), b.close()


def test_minimum(tiny):
    """0 and a minimum past the chunk both feed the ids one at a time."""
    g, _ = tiny
    ids = synth.token_ids(20, synth.TINY.vocab, seed=5)
    rows = []
    for least in (0, 21, None):
        s = g.session(128)
        if least is not None:
            s.set_prefill_batch(least)
        rows.append(_fed(s, [ids]))
        s.close()
    for a, b in zip(rows[0], rows[1]):
        assert np.array_equal(a, b)
    _same_rows(rows[2], rows[0])


@pytest.mark.parametrize("n", [3, 21, 64])
def test_forward(tiny, n):
    """The non-causal forward, whose sessions take the same minimum."""
    g, o = tiny
    ids = synth.token_ids(n, synth.TINY.vocab, seed=60 + n)
    rc, lg = g.forward(ids)
    orc_rc, ref = o.forward(ids)
    assert rc == 0 and orc_rc == 0
    assert max(rel_l2(a, b) for a, b in zip(lg, ref)) < TOL


NARROW = synth.reduced(synth.LLAMA3_8B, dim=512, ffn=1280, n_layers=2, n_heads=8, n_kv_heads=4, vocab=2048, ctx=256)
ONE_TYPE = {Q4_0: synth.reduced(synth.TINY, n_layers=2, vocab=2048), Q4_K: NARROW, Q6_K: NARROW}


@pytest.fixture(scope="module", params=sorted(ONE_TYPE), ids=["q4_0", "q4_k", "q6_k"])
def one_type(request, tmpdir_session):
    """A narrow model whose every matrix is of one type: q/k/v and gate/up in the
    few-row launches that the models above do not reach."""
    t = request.param
    spec = synth.reduced(ONE_TYPE[t], types={r: t for r in list(synth.ROLES) + ["embd", "output"]}, centred=t != Q4_0)
    p = str(tmpdir_session / f"one_type_{t}.gguf")
    synth.write_llama(p, spec, seed=20 + t)
    g, o = GpuModel(p), orc.Model(p)
    yield g, o, spec
    g.close()
    o.close()


@pytest.mark.parametrize("n", [3, 8, 9, 16, 17, 32, 33, 64])
def test_one_type(one_type, n):
    """Against the oracle, and with an f16 cache against the same ids fed one at a
    time (tolerances: test_chunks_of_every_kind)."""
    g, o, spec = one_type
    ids = synth.token_ids(n, spec.vocab, seed=n)
    s, kv = g.session(128), o.kv(128)
    rc, ref = o.prefill(kv, ids)
    assert rc == 0
    _same_rows(_fed(s, [ids]), (ref, *kv.export(n)))
    s.close()
    a, b = g.session(128, kv_f16=True), g.session(128, kv_f16=True)
    b.set_prefill_batch(0)
    _same_rows(_fed(a, [ids]), _fed(b, [ids]), 2.0 ** -8, 2.0 ** -10)
    a.close(), b.close()
