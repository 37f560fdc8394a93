"""matmul_qt of more than 64 rows where the launch plan changes: tiles of 128
rows by 256 outputs in whole rounds of 256, K ranges for all tiles or for those
past the last whole round, ragged last tiles, and the reduce of outputs four at
a time or one (a row count that 4 does not divide).

The check is against float64.  The operands carry 22 bits or more (2^-21
relative per product at most, and 2^-38 of the row's largest activation, whose
scale it shares), the sums are f32: each of the K / 16 matrix instructions, the
few scale steps and the up to 64 partial sums of an output round once."""
from __future__ import annotations

import numpy as np
import pytest

from inferox_amd import synth
from inferox_amd.gguf_writer import Q4_0, Q4_K, Q6_K, Q8_0
from tests.conftest import rel_l2
from tests.gpu_util import GpuModel
from tests.test_gpu_few_rows import _run, _weights
from tests.test_gpu_prefill import TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,m,rows,cols", [
    (Q4_K, 300, 23000, 1024),   # 270 tiles: a whole round, and 14 tiles of 44 rows in 4 ranges
    (Q8_0, 257, 23001, 1024),   # the same with one row in the last tiles, outputs one at a time
    (Q6_K, 100, 301, 4096),     # two tiles in 16 ranges, outputs one at a time
    (Q8_0, 128, 520, 4000),     # 125 steps: a shorter last range
    (Q4_0, 65, 1, 2048),        # one output
    (Q4_K, 129, 256, 256),      # too short to cut: whole tiles, the last of one row
    (Q4_0, 640, 13312, 64),     # 260 whole tiles of two steps
    (Q6_K, 640, 13312, 512),    # four of 260 tiles in 2 ranges of one scale block
])
def test_tiles_and_ranges(t, m, rows, cols):
    w, wf = _weights(t, rows, cols, rows + m)
    a = np.random.default_rng(m).standard_normal((m, cols)).astype(np.float32)
    a[m // 2] = 0.0
    got, a = _run(w, a, rows), a.astype(np.float64)
    bound = (2.0 ** -21 + (cols / 16 + 80) * 2.0 ** -24) * (np.abs(a) @ np.abs(wf).T) + 1e-30
    bound += 2.0 ** -38 * np.outer(np.abs(a).max(axis=1), np.abs(wf).sum(axis=1))
    over = np.abs(got - a @ wf.T) / bound
    assert over.max() <= 1.0, f"{over.max():.2f} of the bound at {np.unravel_index(over.argmax(), over.shape)}"


def test_prompt_of_whole_and_cut_tiles(tmpdir_session):
    """The layer's epilogues (RoPE and cache rows, SwiGLU, residual) through both
    kinds of tiles: 300 ids at the Llama-3-8B width are 336 gate/up tiles, 256
    whole and 80 of 44 rows in ranges, against the ids fed one at a time."""
    spec = synth.reduced(synth.LLAMA3_8B, n_layers=1, ctx=512)
    p = str(tmpdir_session / "l8b_1l_plan.gguf")
    synth.write_llama(p, spec, seed=8)
    g = GpuModel(p)
    ids = synth.token_ids(300, spec.vocab, seed=13)
    a, b = g.session(320), g.session(320)
    b.set_prefill_batch(0)
    (rca, la), (rcb, lb) = a.prefill(ids), b.prefill(ids)
    assert rca == 0 and rcb == 0
    assert max(rel_l2(x, y) for x, y in zip(la, lb)) < TOL
    for x, y in zip(a.kv_export(300), b.kv_export(300)):
        assert rel_l2(x, y) < 1e-4
    a.close(), b.close(), g.close()
