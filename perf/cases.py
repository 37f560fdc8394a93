"""The performance cases: the work a program that uses this library has it do.

Each case is one pass through the public entry points of include/inferox.h,
called through ctypes as inferox_amd._native declares them, on device buffers
that the program owns and on the library's own stream.  The kinds:

  model         a GGUF llama model: prefill of a prompt, then decode steps that
                each return their logits (a chat turn with host-side sampling)
  gemv          y = W x, one decode token through one quantized matrix
  linear        C = A W^T for m tokens (a prompt chunk through one matrix)
  mlp           the feed-forward block of m tokens, composed from operators
  attn_decode   one token's attention over a KV cache
  attn_prefill  a prompt chunk's attention over its own cache rows
  dequant       a GGUF block stream to f32

Shapes are those of the repository's synthetic models (synth.TINY,
synth.LLAMA3_8B, synth.LLAMA3_70B) and, in drawn cases, sizes around them.
Weights are zero-mean random blocks scaled so that a matrix-vector product
keeps the size of its input, as a trained network's do.
"""
import ctypes as C
import math
import os
import tempfile

import numpy as np
import torch

from inferox_amd import _native, synth
from inferox_amd.gguf_writer import F16, F32, Q4_0, Q4_K, Q6_K, Q8_0, GGUFWriter, byte_size

TYPES = {"q4_k": Q4_K, "q6_k": Q6_K, "q8_0": Q8_0, "q4_0": Q4_0, "f16": F16}
EPS = 1e-5


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest model, whole: a short prompt, then a reply of a few
        # tokens; everything is launches and latency
        dict(name="tiny_turn", kind="model", model="tiny", layers=6, prompt=16, steps=8),
        # the 8B layer shape at four layers (of 32; vocabulary 32000), whole: a
        # prompt of 512 ids as one batched prefill, then decode
        dict(name="8b_layers_turn", kind="model", model="llama3-8b", layers=4, prompt=512, steps=8),
        # decode projections of the 8B shape: attention (the smallest call),
        # feed-forward in a Q8_0 file, and the output head (the largest)
        dict(name="gemv_attn_q4k", kind="gemv", type="q4_k", rows=4096, cols=4096),
        dict(name="gemv_ffn_q8", kind="gemv", type="q8_0", rows=14336, cols=4096),
        dict(name="gemv_head_q6k", kind="gemv", type="q6_k", rows=128256, cols=4096),
        # a handful of tokens through one matrix: a very short prompt, the end
        # of a chunked one, a few sequences side by side
        dict(name="linear_8_q4k", kind="linear", type="q4_k", m=8, rows=14336, cols=4096),
        # a long prompt through the same matrix
        dict(name="linear_2048_q4k", kind="linear", type="q4_k", m=2048, rows=14336, cols=4096),
        # the feed-forward block of an ordinary prompt, ragged against every tile
        dict(name="mlp_100", kind="mlp", m=100, dim=4096, ffn=14336),
        # one token over the benchmark's 2048-row cache, and over a long f16 one
        dict(name="attn_decode_2k", kind="attn_decode", kv="f32", rows=2048, heads=32, kv_heads=8, head_dim=128),
        dict(name="attn_decode_8k_f16", kind="attn_decode", kv="f16", rows=8192, heads=64, kv_heads=8, head_dim=128),
        # the attention of a 2048-id prompt
        dict(name="attn_prefill_2k", kind="attn_prefill", kv="f32", n=2048, row0=0, heads=32, kv_heads=8,
             head_dim=128, causal=True),
        # one feed-forward matrix back to f32 (conversion, inspection)
        dict(name="dequant_q4k", kind="dequant", type="q4_k", rows=14336, cols=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["model", "gemv", "gemv", "linear", "linear", "mlp", "attn_decode", "attn_prefill", "dequant"])
    if kind == "model":
        model = rng.choice(["tiny", "llama3-8b"])
        layers = 6 if model == "tiny" else rng.randint(1, 4)
        return dict(kind=kind, model=model, layers=layers, prompt=_log(rng, 2, 512 if model != "tiny" else 200),
                    steps=rng.randint(1, 8))
    if kind in ("gemv", "linear", "dequant"):
        t = rng.choice(["q4_k", "q6_k", "q8_0", "q4_0", "f16"] if kind != "linear" else ["q4_k", "q6_k", "q8_0", "q4_0"])
        cols = 256 * _log(rng, 2, 112) if t in ("q4_k", "q6_k") or rng.random() < 0.5 else 32 * _log(rng, 9, 512)
        rows = _log(rng, 200, 32000)
        rows = max(16, min(rows, (128 << 20) // cols))  # no larger than the head, nor half a GB of f32
        c = dict(kind=kind, type=t, rows=rows, cols=cols)
        if kind == "linear":
            c["rows"] = max(16, min(rows, (58 << 20) // cols))
            c["m"] = _log(rng, 2, 2048)
        return c
    if kind == "mlp":
        dim = 256 * rng.randint(2, 16)
        return dict(kind=kind, m=_log(rng, 2, 512), dim=dim, ffn=256 * _log(rng, dim // 256, dim // 256 * 4))
    kv = rng.choice(["f32", "f16"])
    hd = rng.choice([48, 64, 96, 128, 128])
    kvh = rng.choice([2, 4, 8, 8])
    group = rng.choice([1, 2, 4, 4, 8])
    if kind == "attn_decode":
        return dict(kind=kind, kv=kv, rows=_log(rng, 1, 8448), heads=kvh * group, kv_heads=kvh, head_dim=hd)
    heads = min(kvh * group, 32)
    return dict(kind=kind, kv=kv, n=_log(rng, 16, 2048), row0=rng.choice([0, 0, rng.randint(1, 1024)]),
                heads=heads, kv_heads=kvh, head_dim=hd, causal=rng.random() < 0.8)


# ---------------------------------------------------------------------------
# inputs: random blocks in the GGUF layouts, made on the GPU from the seed
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _half_bytes(x):
    return x.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def _blocks(t, rows, cols, gen, gain=1.0):
    """[n_blocks, block bytes] uint8 on the GPU (F16: [rows, 2 cols]) of a zero-mean
    matrix whose product with a unit-RMS vector has standard deviation `gain`."""
    std = gain / math.sqrt(cols)
    n = rows * cols

    def u8(*shape):
        return torch.randint(0, 256, shape, generator=gen, device="cuda", dtype=torch.uint8)

    def spread(nb):  # block scales around their mean
        return 0.75 + 0.5 * torch.rand(nb, generator=gen, device="cuda")

    if t == F16:
        x = torch.randn(rows, cols, generator=gen, device="cuda") * std
        return x.to(torch.float16).view(torch.uint8)
    if t == Q8_0:  # d, 32 int8
        q = torch.randint(-127, 128, (n // 32, 32), generator=gen, device="cuda", dtype=torch.int8)
        return torch.cat([_half_bytes(spread(n // 32) * (std / 73.3)), q.view(torch.uint8)], 1)
    if t == Q4_0:  # d, 16 bytes of nibbles
        return torch.cat([_half_bytes(spread(n // 32) * (std / 4.64)), u8(n // 32, 16)], 1)
    nb = n // 256
    if t == Q4_K:  # d, dmin, 12 scale bytes, 128 bytes of nibbles; minimum = 7.5 scales: zero mean
        d = spread(nb) * (std / 169.0)
        sc = torch.randint(1, 64, (nb, 8), generator=gen, device="cuda", dtype=torch.int32)
        lo = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
        hi = (sc[:, 4:] & 15) * 17
        s = torch.cat([lo, lo, hi], 1).to(torch.uint8)
        return torch.cat([_half_bytes(d), _half_bytes(7.5 * d), s, u8(nb, 128)], 1)
    if t == Q6_K:  # d, 16 scale bytes, 128 low-nibble bytes, 64 bytes of high bits
        s = torch.randint(1, 8, (nb, 16), generator=gen, device="cuda", dtype=torch.uint8)
        return torch.cat([_half_bytes(spread(nb) * (std / 82.6)), s, u8(nb, 192)], 1)
    raise ValueError(t)


def _hidden(gen, *shape):
    """Activations: unit variance with a few large channels, as a residual stream has."""
    x = torch.randn(*shape, generator=gen, device="cuda")
    x[..., ::97] *= 8.0
    return x


class _Tensor:
    """An uploaded weight matrix."""

    def __init__(self, t, raw, rows, cols):
        host = np.ascontiguousarray(raw.cpu().numpy().reshape(-1))
        self.h = C.c_void_p()
        _native.check(_native.lib().ifx_tensor_upload(t, host.ctypes.data_as(C.c_void_p), host.size, rows, cols,
                                                      C.byref(self.h)), "ifx_tensor_upload")

    def __del__(self):
        if getattr(self, "h", None):
            _native.lib().ifx_tensor_free(self.h)
            self.h = None


class _Model:
    """An opened model and one session."""

    def __init__(self, path, max_seq):
        L = _native.lib()
        self.m, self.s = C.c_void_p(), C.c_void_p()
        _native.check(L.ifx_model_open(path.encode(), C.byref(self.m)), "ifx_model_open")
        _native.check(L.ifx_session_create(self.m, max_seq, C.byref(self.s)), "ifx_session_create")

    def __del__(self):
        if getattr(self, "s", None):
            _native.lib().ifx_session_destroy(self.s)
            self.s = None
        if getattr(self, "m", None):
            _native.lib().ifx_model_close(self.m)
            self.m = None


def _spec(case):
    return synth.reduced(synth.SPECS[case["model"]], n_layers=case["layers"], vocab=32000)


def _model_tensors(case, seed):
    """(name, shape, type, raw bytes on the GPU) of every tensor of the model, one at a time."""
    spec = _spec(case)
    for i, (name, shape, t, rows, cols) in enumerate(spec.shapes()):
        g = _gen(seed * 1000003 + i)
        if t == F32:
            yield name, shape, t, (1.0 + 0.02 * torch.randn(cols, generator=g, device="cuda")).view(torch.uint8)
        else:
            gain = {"embd": math.sqrt(cols), "output": 2.0, "q": 1.25, "k": 1.25}.get(synth.role_of(name), 1.0)
            yield name, shape, t, _blocks(t, rows, cols, g, gain)


def _model_ids(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    return r.randint(0, 32000, case["prompt"] + case["steps"]).astype(np.uint32)


def _mlp_inputs(case, seed):
    g = _gen(seed)
    m, d, f = case["m"], case["dim"], case["ffn"]
    return (_hidden(g, m, d), 1.0 + 0.02 * torch.randn(d, generator=g, device="cuda"),
            _blocks(Q4_K, f, d, g), _blocks(Q4_K, f, d, g), _blocks(Q6_K, d, f, g))


def _attn_inputs(case, seed):
    """q, and the caches [kv_heads][max_seq][head_dim] with some rows past those attended."""
    g = _gen(seed)
    kvh, hd, h = case["kv_heads"], case["head_dim"], case["heads"]
    n = case["rows"] if case["kind"] == "attn_decode" else case["row0"] + case["n"]
    max_seq = n + 64
    dt = torch.float16 if case["kv"] == "f16" else torch.float32
    k = torch.randn(kvh, max_seq, hd, generator=g, device="cuda").to(dt)
    v = torch.randn(kvh, max_seq, hd, generator=g, device="cuda").to(dt)
    nq = 1 if case["kind"] == "attn_decode" else case["n"]
    q = torch.randn(nq, h * hd, generator=g, device="cuda") * 1.5
    return q, k, v, max_seq


def _p(t):
    return C.c_void_p(t.data_ptr())


def _np(a):
    return a.ctypes.data_as(C.c_void_p)


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    L, kind = _native.lib(), case["kind"]
    s = {"L": L, "case": case}
    if kind == "model":
        spec = _spec(case)
        w = GGUFWriter()
        w.add_string("general.architecture", "llama").add_u32("llama.vocab_size", spec.vocab)
        w.add_u32("llama.embedding_length", spec.dim).add_u32("llama.block_count", spec.n_layers)
        w.add_u32("llama.attention.head_count", spec.n_heads).add_u32("llama.attention.head_count_kv", spec.n_kv_heads)
        w.add_u32("llama.feed_forward_length", spec.ffn).add_f32("llama.attention.layer_norm_rms_epsilon", EPS)
        w.add_f32("llama.rope.freq_base", spec.rope_theta).add_u32("llama.context_length", 4096)
        for name, shape, t, raw in _model_tensors(case, seed):
            host = raw.cpu().numpy().reshape(-1)
            w.add_tensor(name, shape, t, fill=lambda view, host=host: np.copyto(view, host))
        with tempfile.TemporaryDirectory() as d:
            path = os.path.join(d, "m.gguf")
            w.write(path)
            s["model"] = _Model(path, case["prompt"] + case["steps"] + 32)
        s["ids"] = _model_ids(case, seed)
        s["logits"] = np.empty((case["steps"], spec.vocab), np.float32)
    elif kind in ("gemv", "linear"):
        g, t = _gen(seed), TYPES[case["type"]]
        m = case.get("m", 1)
        s["x"] = _hidden(g, m, case["cols"])
        s["w"] = _Tensor(t, _blocks(t, case["rows"], case["cols"], g), case["rows"], case["cols"])
        s["y"] = torch.empty(m, case["rows"], device="cuda")
    elif kind == "mlp":
        x, nw, gate, up, down = _mlp_inputs(case, seed)
        m, d, f = case["m"], case["dim"], case["ffn"]
        s.update(x=x, nw=nw, gate=_Tensor(Q4_K, gate, f, d), up=_Tensor(Q4_K, up, f, d), down=_Tensor(Q6_K, down, d, f))
        s.update(xn=torch.empty_like(x), g=torch.empty(m, f, device="cuda"), u=torch.empty(m, f, device="cuda"),
                 y=torch.empty_like(x))
    elif kind in ("attn_decode", "attn_prefill"):
        s["q"], s["k"], s["v"], s["max_seq"] = _attn_inputs(case, seed)
        s["y"] = torch.empty_like(s["q"])
    else:
        t = TYPES[case["type"]]
        s["raw"] = _blocks(t, case["rows"], case["cols"], _gen(seed)).reshape(-1)
        s["y"] = torch.empty(case["rows"], case["cols"], device="cuda")
    torch.cuda.synchronize()  # the library works on a stream of its own
    return s


def run(s):
    L, c = s["L"], s["case"]
    kind, ck = c["kind"], _native.check
    if kind == "model":
        ses, ids, n = s["model"].s, s["ids"], c["prompt"]
        ck(L.ifx_session_clear(ses), "ifx_session_clear")
        ck(L.ifx_prefill(ses, _np(ids), n, None), "ifx_prefill")
        for i in range(c["steps"]):
            ck(L.ifx_decode_step(ses, int(ids[n + i]), _np(s["logits"][i])), "ifx_decode_step")
        return s["logits"]
    if kind == "gemv":
        ck(L.ifx_gemv(s["w"].h, _p(s["x"]), _p(s["y"]), None), "ifx_gemv")
    elif kind == "linear":
        ck(L.ifx_matmul_qt(_p(s["x"]), c["m"], s["w"].h, _p(s["y"]), None), "ifx_matmul_qt")
    elif kind == "mlp":
        m, d, f = c["m"], c["dim"], c["ffn"]
        ck(L.ifx_memcpy_d2d(_p(s["xn"]), _p(s["x"]), m * d * 4), "ifx_memcpy_d2d")  # the norm works in place
        ck(L.ifx_ops_rms_norm_rows(_p(s["xn"]), _p(s["nw"]), d, m, EPS, None), "ifx_ops_rms_norm_rows")
        ck(L.ifx_matmul_qt(_p(s["xn"]), m, s["gate"].h, _p(s["g"]), None), "ifx_matmul_qt")
        ck(L.ifx_matmul_qt(_p(s["xn"]), m, s["up"].h, _p(s["u"]), None), "ifx_matmul_qt")
        ck(L.ifx_ops_swiglu(_p(s["g"]), _p(s["u"]), _p(s["g"]), m * f, None), "ifx_ops_swiglu")
        ck(L.ifx_matmul_qt(_p(s["g"]), m, s["down"].h, _p(s["y"]), None), "ifx_matmul_qt")
        ck(L.ifx_ops_add_in_place(_p(s["y"]), _p(s["x"]), m * d, None), "ifx_ops_add_in_place")
    elif kind == "attn_decode":
        ck(L.ifx_ops_attention_decode(_p(s["q"]), _p(s["k"]), _p(s["v"]), int(c["kv"] == "f16"), s["max_seq"],
                                      c["rows"], c["heads"], c["kv_heads"], c["head_dim"], _p(s["y"]), None),
           "ifx_ops_attention_decode")
    elif kind == "attn_prefill":
        ck(L.ifx_ops_attention_prefill(_p(s["q"]), _p(s["k"]), _p(s["v"]), int(c["kv"] == "f16"), s["max_seq"],
                                       c["row0"], c["n"], c["heads"], c["kv_heads"], c["head_dim"],
                                       int(c["causal"]), _p(s["y"]), None), "ifx_ops_attention_prefill")
    else:
        n = c["rows"] * c["cols"]
        ck(L.ifx_dequantize_f32(TYPES[c["type"]], n, _p(s["raw"]), s["raw"].numel(), _p(s["y"]), n, None),
           "ifx_dequantize_f32")
    return s["y"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "model":
        spec, n, k = _spec(case), case["prompt"], case["steps"]
        layer = sum(byte_size(t, r * c) for (nm, _, t, r, c) in spec.shapes() if nm.startswith("blk."))
        params = sum(r * c for (nm, _, t, r, c) in spec.shapes() if nm.startswith("blk.") and t != F32)
        head = byte_size(spec.t("output"), spec.vocab * spec.dim)
        kv_row = 2 * spec.n_layers * spec.kv_dim * 4
        kv = kv_row * (n + sum(n + i + 1 for i in range(k)))
        att = 4 * spec.n_layers * spec.dim * (n * (n + 1) // 2 + sum(n + i + 1 for i in range(k)))
        return {"bytes": layer * (1 + k) + head * (1 + k) + kv + k * spec.vocab * 4,
                "flops": 2 * params * (n + k) + 2 * spec.vocab * spec.dim * (1 + k) + att}
    if kind in ("gemv", "linear"):
        m, r, c = case.get("m", 1), case["rows"], case["cols"]
        return {"bytes": byte_size(TYPES[case["type"]], r * c) + 4 * m * (r + c), "flops": 2 * m * r * c}
    if kind == "mlp":
        m, d, f = case["m"], case["dim"], case["ffn"]
        return {"bytes": 2 * byte_size(Q4_K, d * f) + byte_size(Q6_K, d * f) + 8 * m * d, "flops": 6 * m * d * f}
    es, kvd, qd = (2 if case.get("kv") == "f16" else 4), 0, 0
    if kind != "dequant":
        kvd, qd = case["kv_heads"] * case["head_dim"], case["heads"] * case["head_dim"]
    if kind == "attn_decode":
        return {"bytes": 2 * case["rows"] * kvd * es + 8 * qd, "flops": 4 * case["rows"] * qd}
    if kind == "attn_prefill":
        n = case["n"]
        pairs = n * (n + 1) // 2 if case["causal"] else n * n
        return {"bytes": 2 * n * kvd * es + 8 * n * qd, "flops": 4 * pairs * qd}
    n = case["rows"] * case["cols"]
    return {"bytes": byte_size(TYPES[case["type"]], n) + 4 * n, "flops": 0}


def tolerance(case):
    # f32 sums of operands carried at 22 bits or more, measured against exact():
    # 2e-7 to 7e-7 of the result's norm; whole models 1e-6 to 2e-6, and as much
    # again between two runs (partial sums added in another order)
    if case["kind"] == "dequant":
        return "exact"
    if case["kind"] == "model":
        return {"rel": 2e-5, "max": 4e-4}
    return {"rel": 4e-6, "max": 1e-4}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _dequant(t, raw, rows, cols):
    """GGUF blocks (the reference's layouts) as a float64 [rows, cols] matrix."""
    def half(lo, n=1):
        return b[:, lo:lo + 2 * n].contiguous().view(torch.float16).double()

    if t == F16:
        return raw.contiguous().view(torch.float16).double().reshape(rows, cols)
    if t == Q8_0:
        b = raw.reshape(-1, 34)
        return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)
    if t == Q4_0:
        b = raw.reshape(-1, 18)
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8
        return (half(0) * q).reshape(rows, cols)
    if t == Q4_K:
        b = raw.reshape(-1, 144)
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = torch.stack([b[:, 16:] & 15, b[:, 16:] >> 4], 2).reshape(-1, 8, 32).double()
        w = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
        return w.reshape(rows, cols)
    b = raw.reshape(-1, 210)
    lo = torch.stack([b[:, 18:146] & 15, b[:, 18:146] >> 4], 2).reshape(-1, 256)
    h = b[:, 146:]
    hi = torch.stack([h & 3, (h >> 2) & 3, (h >> 4) & 3, h >> 6], 2).reshape(-1, 256)
    q = (lo | (hi << 4)).double().reshape(-1, 16, 16) - 32
    return ((half(0) * b[:, 2:18].double())[:, :, None] * q).reshape(rows, cols)


def _times(x, t, raw, rows, cols):
    """x W^T in 64 bits, some rows of W at a time."""
    raw = raw.reshape(rows, -1)
    step = max(1, (1 << 27) // cols)
    return torch.cat([x @ _dequant(t, raw[r:r + step], min(step, rows - r), cols).T for r in range(0, rows, step)], 1)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _silu(g):
    return g / (1 + torch.exp(-g))


def _attend(q, k, v, first, causal):
    """q [n, heads, hd] against k, v [rows, kv_heads, hd]: query t sees rows 0 .. first + t
    (causal), or all."""
    n, h, hd = q.shape
    group = h // k.shape[1]
    out = torch.empty_like(q)
    seen = torch.arange(k.shape[0], device=q.device)[None, :] <= first + torch.arange(n, device=q.device)[:, None]
    for i in range(h):
        s = q[:, i] @ k[:, i // group].T.contiguous() / math.sqrt(hd)
        if causal:
            s = s.masked_fill(~seen, -math.inf)
        out[:, i] = torch.softmax(s, -1) @ v[:, i // group]
    return out


def _rotate(x, pos, theta):
    """RoPE on adjacent pairs of [n, heads, hd]; the angles are f32, as the format defines them."""
    hd = x.shape[-1]
    inv = (np.float32(1) / np.power(np.float32(theta), np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd),
                                    dtype=np.float32)).astype(np.float32)
    ang = (np.asarray(pos, np.float32)[:, None] * inv).astype(np.float64)
    cos, sin = (torch.from_numpy(f(ang)).to(x.device)[:, None, :] for f in (np.cos, np.sin))
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x.shape)


def _exact_model(case, seed):
    spec, n, steps = _spec(case), case["prompt"], case["steps"]
    ten = {name: (t, raw) for name, _, t, raw in _model_tensors(case, seed)}
    ids = torch.from_numpy(_model_ids(case, seed).astype(np.int64)).cuda()
    D, hd, nh, kvh = spec.dim, spec.head_dim, spec.n_heads, spec.n_kv_heads
    # the session's default positions: 0 .. n - 1 for the prompt, 0 for each decoded token
    pos = list(range(n)) + [0] * steps
    emb = ten["token_embd.weight"]
    x = _dequant(emb[0], emb[1].reshape(spec.vocab, -1)[ids], n + steps, D)

    def vec(name):
        return ten[name][1].view(torch.float32).double()

    def mat(x, name, rows, cols):
        return _times(x, *ten[name], rows, cols)

    for i in range(spec.n_layers):
        p = "blk.%d." % i
        y = _norm(x, vec(p + "attn_norm.weight"))
        q = _rotate(mat(y, p + "attn_q.weight", D, D).reshape(-1, nh, hd), pos, spec.rope_theta)
        k = _rotate(mat(y, p + "attn_k.weight", spec.kv_dim, D).reshape(-1, kvh, hd), pos, spec.rope_theta)
        v = mat(y, p + "attn_v.weight", spec.kv_dim, D).reshape(-1, kvh, hd)
        x = x + mat(_attend(q, k, v, 0, True).reshape(-1, D), p + "attn_output.weight", D, D)
        y = _norm(x, vec(p + "ffn_norm.weight"))
        y = _silu(mat(y, p + "ffn_gate.weight", spec.ffn, D)) * mat(y, p + "ffn_up.weight", spec.ffn, D)
        x = x + mat(y, p + "ffn_down.weight", D, spec.ffn)
    x = _norm(x[n:], vec("output_norm.weight"))
    return mat(x, "output.weight", spec.vocab, D).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _exact_model(case, seed)
    if kind in ("gemv", "linear"):
        g, t = _gen(seed), TYPES[case["type"]]
        x = _hidden(g, case.get("m", 1), case["cols"]).double()
        return _times(x, t, _blocks(t, case["rows"], case["cols"], g), case["rows"], case["cols"])
    if kind == "mlp":
        x, nw, gate, up, down = _mlp_inputs(case, seed)
        d, f = case["dim"], case["ffn"]
        x = x.double()
        y = _norm(x, nw.double())
        y = _silu(_times(y, Q4_K, gate, f, d)) * _times(y, Q4_K, up, f, d)
        return _times(y, Q6_K, down, d, f) + x
    if kind in ("attn_decode", "attn_prefill"):
        q, k, v, _ = _attn_inputs(case, seed)
        lo, n = (0, case["rows"]) if kind == "attn_decode" else (case["row0"], case["n"])
        k, v = (x[:, lo:lo + n].transpose(0, 1).double().contiguous() for x in (k, v))
        y = _attend(q.double().reshape(q.shape[0], case["heads"], -1), k, v, 0,
                    kind == "attn_prefill" and case["causal"])
        return y.reshape(q.shape)
    t = TYPES[case["type"]]
    return _dequant(t, _blocks(t, case["rows"], case["cols"], _gen(seed)), case["rows"], case["cols"])
