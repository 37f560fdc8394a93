"""The library's host code on a device whose memory runs out, on the CPU: a
simulated runtime (tests/hostsim/hip_sim.cpp) takes the HIP runtime's place in a
process of its own, fails allocations past a set size, and counts launches
without running them. What a call returns, how much stays allocated after it and
which kernels it launched are checked; results are not computed."""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "inferox_amd", "lib", "libinferox.so")

HEAD = """
import ctypes as C, sys
sim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library: its symbols win
sim.sim_used.restype = C.c_size_t
sim.sim_limit.argtypes = [C.c_size_t]
sim.sim_launches.restype = C.c_long
from inferox_amd import _native, synth
from inferox_amd.gguf_writer import Q4_K
from tests.gpu_util import Dev, GpuModel, Tensor
import numpy as np
L = _native.lib()
OK = 0
MB = 1 << 20
SPEC = synth.reduced(synth.LLAMA3_8B, dim=512, ffn=1024, n_layers=2, n_heads=8, n_kv_heads=4, vocab=4096)
def used(): return sim.sim_used()
def room(n): sim.sim_limit(used() + n)
def plenty(): sim.sim_limit(8 << 30)
def launches(part): return sim.sim_launches(part.encode())
def model():
    synth.write_llama(sys.argv[2], SPEC, seed=1)
    return GpuModel(sys.argv[2])
ids = synth.token_ids(300, SPEC.vocab, seed=2)
"""


@pytest.fixture(scope="module")
def sim(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx or not os.path.exists(LIB):
        pytest.skip("needs g++ and the built library")
    out = str(tmp_path_factory.mktemp("hostsim") / "hip_sim.so")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        "-w", os.path.join(ROOT, "tests", "hostsim", "hip_sim.cpp"), "-o", out],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    return out


def _run(sim, tmp_path, body):
    r = subprocess.run([sys.executable, "-c", HEAD + body, sim, str(tmp_path / "m.gguf")], cwd=ROOT,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout


def test_a_long_prompt_without_room_strands_nothing(sim, tmp_path):
    """A prompt too long for the memory left fails and leaves what it found; the
    short prompts after it still run layer by layer."""
    _run(sim, tmp_path, """
g = model()
s = g.session(400)
assert s.prefill(ids[:10], False)[0] == OK
assert launches("k_skinny_qkv") == 2
first = used()
for k in range(3):
    s.clear()
    room(40 * MB)
    rc, _ = s.prefill(ids, False)
    assert rc != OK
    assert len(s) == 0
    assert s.prefill(ids[:10], False)[0] == OK
    assert launches("k_skinny_qkv") == 4 + 2 * k
    assert used() <= first, (used(), first)
plenty()
s.clear()
assert s.prefill(ids, False)[0] == OK
s.clear()
assert s.prefill(ids[:10], False)[0] == OK
s.close(); g.close()
assert used() == 0, used()
""")


def test_kept_workspaces_make_room(sim, tmp_path):
    """What operators keep between calls goes to whoever finds no memory left: a
    buffer, a matrix, a session, a prompt's workspace, another operator."""
    _run(sim, tmp_path, """
raw = synth.random_centred_blocks(Q4_K, 1024 * 512, 512, "q", 1)
w = Tensor(Q4_K, raw, 1024, 512)
x, q, cache = Dev(4 * 300 * 1024), Dev(4 * 32 * 128), Dev(4 * 8 * 3100 * 128)
def keep():
    plenty()
    had = used()
    assert L.ifx_matmul_qt(x.ptr, 300, w.h, x.ptr, None) == OK
    assert L.ifx_ops_attention_decode(q.ptr, cache.ptr, cache.ptr, 0, 3100, 3000, 32, 8, 128, q.ptr, None) == OK
    kept = used() - had
    assert kept >= 2 * MB, kept
    return kept

kept = keep()
room(0)
d = Dev(kept)                      # all of it
assert L.ifx_gemv(w.h, x.ptr, x.ptr, None) == OK   # the failed attempt left no error behind
d.free()

keep()
room(0)
w2 = Tensor(Q4_K, raw, 1024, 512)

plenty()
g = model()
keep()
room(256 << 10)
s = g.session(16)                  # a megabyte or so

plenty()
s2 = g.session(128)
s2.prefill(ids[:70], False)        # has its own workspace
keep()
room(0)
s2.clear()
assert s2.prefill(ids[:71], False)[0] == OK

keep()
room(0)
assert L.ifx_matmul_qt(x.ptr, 290, w.h, x.ptr, C.c_void_p(8)) == OK  # a caller's stream: a workspace of its own
assert L.ifx_ops_attention_decode(q.ptr, cache.ptr, cache.ptr, 0, 3100, 3000, 32, 8, 128, q.ptr, None) == OK
""")


def test_logits_without_room(sim, tmp_path):
    """The logits of every row of a short prompt, where there is no memory for
    them: the ids are fed one at a time. Of a long one: an error before anything
    is queued, and the session goes on as it was."""
    _run(sim, tmp_path, """
g = model()
s = g.session(400)
assert s.prefill(ids[:10], False)[0] == OK
few, steps = launches("k_skinny_qkv"), launches("k_finalize")
sim.sim_limit(0)
assert s.prefill(ids[:10], True)[0] == OK
assert len(s) == 20 and launches("k_skinny_qkv") == few and launches("k_finalize") == steps + 10
plenty()
assert s.prefill(ids[:200], False)[0] == OK
steps, states = launches("k_finalize"), launches("k_state")
sim.sim_limit(0)
assert s.prefill(ids[:100], True)[0] != OK
assert len(s) == 220 and launches("k_finalize") == steps and launches("k_state") == states
plenty()
assert s.prefill(ids[:100], True)[0] == OK
assert len(s) == 320
assert g.forward(ids[:10])[0] == OK
""")


def test_short_prompt_launches(sim, tmp_path):
    """A short prompt with every row's logits: the few-row launches from the layers
    to the output head, none of the tile GEMMs' (128 rows, whatever the ids)."""
    _run(sim, tmp_path, """
g = model()
s = g.session(64)
assert s.prefill(ids[:3], True)[0] == OK
assert launches("k_skinny_qkv") == 2 and launches("k_gemm_skinny") == 5
assert launches("k_prep_rows") == 0
""")
