"""Prefill attention on both sides of its launch rule: 64 heads are 192
workgroups of 128 queries at 384 rows (fewer than the 256 that fill the chip:
the workgroups of 64 queries whose waves halve each block's keys) and 256 at 385
and 449 rows (the last query block of one row, and of 65).  Against float64, at
the bar of tests/test_gpu_attention.py; and the first 384 rows of a causal
chunk, which both kernels attend alike, within twice it of each other."""
from __future__ import annotations

import numpy as np
import pytest

from inferox_amd import _native
from tests.gpu_util import Dev
from tests.test_gpu_attention import KV_F16, KV_F32, TOL_PRE, head_major, prefill64, prefill_case

pytestmark = pytest.mark.gpu

NH, NKV = 64, 8


def _run(q, k, v, n, hd, causal, f16):
    dk, dv = (Dev.of(head_major(x[:n], n, NKV, hd, n + 5, f16)) for x in (k, v))
    dq, do = Dev.of(np.ascontiguousarray(q[:n])), Dev(n * NH * hd * 4)
    rc = _native.lib().ifx_ops_attention_prefill(dq.ptr, dk.ptr, dv.ptr, KV_F16 if f16 else KV_F32, n + 5, 0, n, NH,
                                                 NKV, hd, int(causal), do.ptr, None)
    assert rc == 0
    return do.get(np.float32, n * NH * hd).reshape(n, NH, hd).astype(np.float64)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("hd", [48, 64, 96, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_both_sides(hd, causal, f16):
    q, k, v = prefill_case(449, NH, NKV, hd, seed=hd, f16=f16)
    rows = [0, 31, 32, 63, 64, 127, 128, 200, 383]
    outs = {}
    for n in (384, 385, 449):
        got = outs[n] = _run(q, k, v, n, hd, causal, f16)
        assert np.isfinite(got).all()
        pick = rows + [n - 1]
        ref, scale = prefill64(q[:n], k[:n], v[:n], pick, NH, NKV, hd, causal)
        assert (np.linalg.norm(got[pick] - ref, axis=2) / scale).max() <= TOL_PRE, n
    if causal:
        vmag = np.linalg.norm(v.reshape(449, NKV, hd), axis=2).max()
        assert np.abs(outs[384] - outs[385][:384]).max() <= 2 * TOL_PRE * vmag
