"""What a program built on this library has it do, as cases that can be timed
and compared: captured decode and verify steps, prefill of short and long
prompts, the two lm_heads, one bare projection call, and the load of a fused
projection.

    listed()              the cases that stand for the range
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   weights, inputs, buffers and captured graph of a program
    run(state)            one pass through the public entry points
    work(case)            bytes and operations that a pass cannot do without
    tolerance(case)       how far another correct implementation may be off
    exact(case, seed)     the outputs of the same inputs in 64 bits

Weights are INT4 group-128 with random levels, zero points around the middle
and scales that keep the outputs of a projection near 1; activations are normal
with a spread between channels, as hidden states have it. Programs capture
their decode, verify and short-prompt steps in a graph (rows <= GRAPH_ROWS) and
launch longer prompts eagerly.
"""
from __future__ import annotations

import math
import os
import sys
import weakref

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "qwen38-3090-cuda-server_amd"))

import w4a16_hip as hip  # noqa: E402

EPS = 1e-6
GROUP = 128
GRAPH_ROWS = 256            # steps of at most this many rows are captured
SKINNY_ROWS = 16            # rows of the decode / verify entry points
EMB = 8192                  # rows of the embedding table the step reads from
WORKSPACE = 256 << 20       # the reference's prefill workspace

# (hidden, qkv rows, attention width, intermediate): the benchmark's layer, the
# reference model's two layer kinds, and the 2-, 4- and 8-way shards.
LAYER = (5120, 7168, 4096, 17408)
LAYERS = (LAYER, (5120, 16384, 6144, 17408), (5120, 14336, 6144, 17408),
          (5120, 3584, 2048, 8704), (5120, 1792, 1024, 4352), (5120, 896, 512, 2176))
VOCAB = 248320


def _layer(name, rows, layers, dims):
    return {"name": name, "op": "layers", "rows": rows, "layers": layers, "hidden": dims[0],
            "qkv": dims[1], "attn": dims[2], "inter": dims[3]}


def listed():
    return [
        # one projection called on its own: k_proj of one token, nothing captured
        {"name": "call_k_proj", "op": "call", "n": 1024, "k": 5120, "f32": False},
        # one decoded token through a stretch of layers (the benchmark's shapes)
        _layer("decode", 1, 4, LAYER),
        # the same on one of eight GPUs: small, latency-bound projections
        _layer("decode_shard8", 1, 8, LAYERS[5]),
        # speculative verify: the last token and eight drafts
        _layer("verify_9", 9, 2, LAYER),
        # the widest verify, over the reference model's other layer kind
        _layer("verify_16_mix", 16, 2, LAYERS[1]),
        # greedy verify over the INT4 head: no logits are wanted
        {"name": "head4_greedy_9", "op": "head", "bits": 4, "rows": 9, "vocab": VOCAB, "hidden": 5120,
         "logits": False},
        # the default 8-bit head of a short verify, with the logits a sampler reads
        {"name": "head8_logits_5", "op": "head", "bits": 8, "rows": 5, "vocab": VOCAB, "hidden": 5120,
         "logits": True},
        # prompts: a few dozen tokens, a chat turn, a ragged chunk, a full chunk
        _layer("prefill_33", 33, 1, LAYER),
        _layer("prefill_200", 200, 1, LAYER),
        _layer("prefill_1000", 1000, 1, LAYER),
        _layer("prefill_4096", 4096, 1, LAYER),
        # a checkpoint's q, k and v repacked into one weight, and its rows read
        # back as bf16 (the loader's check)
        {"name": "load_qkv", "op": "load", "k": 5120, "n0": 5120, "n1": 1024, "n2": 1024},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_dims(rng):
    if rng.random() < 0.6:
        return rng.choice(LAYERS)
    return (128 * rng.randint(8, 48), 64 * rng.randint(9, 150), 128 * rng.randint(4, 48),
            128 * rng.randint(8, 140))


def draw(rng):
    r = rng.random()
    if r < 0.4:
        dims = _draw_dims(rng)
        rows = 1 if rng.random() < 0.35 else rng.randint(2, SKINNY_ROWS)
        c = _layer("", rows, rng.randint(2, 4), dims)
    elif r < 0.75:
        dims = _draw_dims(rng)
        # the full chunk over the widest layers stays below the listed one
        c = _layer("", _log_int(rng, SKINNY_ROWS + 1, 4000 if dims[1] <= 7168 else 3000), 1, dims)
    elif r < 0.87:
        c = {"op": "head", "bits": rng.choice((4, 8)), "rows": rng.randint(1, SKINNY_ROWS),
             "vocab": 64 * _log_int(rng, 485, VOCAB // 64), "hidden": rng.choice((2560, 4096, 5120)),
             "logits": rng.random() < 0.5}
    elif r < 0.94:
        c = {"op": "call", "n": 64 * _log_int(rng, 2, 544), "k": 128 * _log_int(rng, 2, 136),
             "f32": rng.random() < 0.3}
    else:
        c = {"op": "load", "k": 128 * rng.randint(8, 136), "n0": 64 * rng.randint(8, 100),
             "n1": 64 * rng.randint(1, 40), "n2": 64 * rng.randint(1, 40)}
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs
class State:
    """What the program keeps: device buffers, weights and the captured step.
    The library's allocations are given back with the state."""

    def __init__(self):
        self.graph = None
        self._owned = []
        weakref.finalize(self, State._release, self._owned)

    @staticmethod
    def _release(owned):
        for free, handle in owned:
            free(handle)
        owned.clear()

    def own(self, free, handle):
        self._owned.append((free, handle))
        return handle


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _bf16(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)


def _hidden(g, rows, dim):
    """Hidden states: normal, with channels of different size."""
    spread = torch.exp(0.5 * torch.randn(dim, generator=g, device="cuda"))
    x = torch.randn(rows, dim, generator=g, device="cuda") * spread
    return x.to(torch.bfloat16)


def _int4(g, n, k):
    """compressed-tensors source of one projection: packed [n][k/8], scale
    [n][G] bf16, zero points [n/8][G]."""
    G = k // GROUP
    i32 = dict(generator=g, device="cuda", dtype=torch.int32)
    packed = torch.randint(-(1 << 31), (1 << 31) - 1, (n, k // 8), **i32)
    zp = (torch.randint(0, (1 << 31) - 1, (n // 8, G), **i32) & 0x77777777) + 0x44444444
    scale = ((0.5 + torch.rand(n, G, generator=g, device="cuda")) * (0.19 / math.sqrt(k))).to(torch.bfloat16)
    return packed, scale, zp


def _weight(st, g, n, k):
    packed, scale, zp = _int4(g, n, k)
    w = hip.awq_alloc_fused(n, k)
    st.own(hip.awq_free, w)
    hip.awq_repack_into(w, 0, packed, scale, zp, n)
    return w


def _layer_inputs(g, c, weight):
    """One layer's norm weights, attention outputs and projections, in the order
    the generator gives them."""
    h, m = c["hidden"], c["rows"]
    return {
        "n1": 0.1 * _bf16(g, h), "n2": 0.1 * _bf16(g, h), "attn": _bf16(g, m, c["attn"]),
        "qkv": weight(g, c["qkv"], h), "o": weight(g, h, c["attn"]),
        "gu": weight(g, 2 * c["inter"], h), "down": weight(g, h, c["inter"]),
    }


def _empty(*shape, dtype=torch.bfloat16):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _embedding(g, c):
    table = _hidden(g, EMB, c["hidden"])
    ids = torch.randint(0, EMB, (c["rows"],), generator=g, device="cuda")
    return table, ids


def prepare(case, seed):
    c = dict(case)
    st = State()
    st.case = c
    g = _gen(seed)
    if c["op"] == "call":
        st.w = _weight(st, g, c["n"], c["k"])
        st.x = _hidden(g, 1, c["k"])
        st.y = _empty(1, c["n"], dtype=torch.float32 if c["f32"] else torch.bfloat16)
        st.scratch = st.own(hip.gemv_scratch_free, hip.gemv_scratch_alloc(c["k"], c["n"], GROUP, 1))
    elif c["op"] == "layers":
        _prepare_layers(st, g, c)
    elif c["op"] == "head":
        _prepare_head(st, g, c)
    else:
        k = c["k"]
        st.parts = [_int4(g, n, k) for n in _parts(c)]
        st.w = st.own(hip.awq_free, hip.awq_alloc_fused(sum(_parts(c)), k))
        st.rows = _empty(sum(_parts(c)), k)
    torch.cuda.synchronize()
    return st


def _parts(c):
    return [c["n0"], c["n1"], c["n2"]]


def _prepare_layers(st, g, c):
    h, m, inter = c["hidden"], c["rows"], c["inter"]
    st.table, st.ids = _embedding(g, c)
    st.layers = [_layer_inputs(g, c, lambda g_, n, k: _weight(st, g_, n, k)) for _ in range(c["layers"])]
    st.h, st.norm = _empty(m, h), _empty(m, h)
    st.qkv = [_empty(m, c["qkv"]) for _ in range(c["layers"])]
    st.gu, st.act, st.proj = _empty(m, 2 * inter), _empty(m, inter), _empty(m, h)
    st.scratch = st.own(hip.gemv_scratch_free, hip.gemv_scratch_alloc(
        max(h, c["attn"], inter), max(h, c["qkv"], 2 * inter), GROUP, SKINNY_ROWS))
    st.ws = None
    if m > SKINNY_ROWS:
        st.ws = st.own(hip.gemm_workspace_free, hip.gemm_workspace_alloc(WORKSPACE))
    if m <= GRAPH_ROWS:
        torch.cuda.synchronize()
        st.graph = torch.cuda.CUDAGraph()
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            st.graph.capture_begin()
            _step(st)
            st.graph.capture_end()


def _prepare_head(st, g, c):
    n, k, m = c["vocab"], c["hidden"], c["rows"]
    st.h, st.nw, st.norm = _hidden(g, m, k), 0.1 * _bf16(g, k), _empty(m, k)
    if c["bits"] == 4:
        st.w = _weight(st, g, n, k)
    else:
        src = _head_rows(g, n, k)
        st.w = st.own(hip.w8a16_free, hip.quantize_w8a16(src, n, k))
        torch.cuda.synchronize()
    st.logits = _empty(m, n) if c["logits"] else None
    st.idx = _empty(m, dtype=torch.int32)
    st.scratch = st.own(hip.gemv_scratch_free, hip.gemv_scratch_alloc(k, n, GROUP, SKINNY_ROWS))


def _head_rows(g, n, k):
    return (torch.randn(n, k, generator=g, device="cuda", dtype=torch.bfloat16)) * (1.0 / math.sqrt(k))


# --------------------------------------------------------------------- run
def _step(st):
    c = st.case
    m, h, inter = c["rows"], c["hidden"], c["inter"]
    torch.index_select(st.table, 0, st.ids, out=st.h)
    for layer, qkv in zip(st.layers, st.qkv):
        if m <= SKINNY_ROWS:
            hip.gemv_rmsnorm_w4a16(qkv, layer["qkv"], st.h, layer["n1"], EPS, m, st.scratch, tmp=st.norm)
            hip.gemv_residual_w4a16(st.h, layer["o"], layer["attn"], m, st.scratch)
            hip.rmsnorm(st.norm, st.h, layer["n2"], m, h, EPS)
            hip.gemv_swiglu_w4a16(st.act, layer["gu"], st.norm, m, st.scratch, tmp=st.gu)
            hip.gemv_residual_w4a16(st.h, layer["down"], st.act, m, st.scratch)
        else:
            hip.rmsnorm(st.norm, st.h, layer["n1"], m, h, EPS)
            hip.linear_w4a16(qkv, layer["qkv"], st.norm, m, st.scratch, st.ws)
            hip.linear_w4a16(st.proj, layer["o"], layer["attn"], m, st.scratch, st.ws)
            hip.residual_add(st.h, st.proj, m * h)
            hip.rmsnorm(st.norm, st.h, layer["n2"], m, h, EPS)
            hip.linear_w4a16(st.gu, layer["gu"], st.norm, m, st.scratch, st.ws)
            hip.swiglu(st.act, st.gu, m, inter)
            hip.linear_w4a16(st.proj, layer["down"], st.act, m, st.scratch, st.ws)
            hip.residual_add(st.h, st.proj, m * h)


def run(state):
    st, c = state, state.case
    if c["op"] == "call":
        (hip.gemv_w4a16_f32 if c["f32"] else hip.gemv_w4a16)(st.y, st.w, st.x, st.scratch)
        return st.y
    if c["op"] == "layers":
        if st.graph is not None:
            st.graph.replay()
        else:
            _step(st)
        return {"qkv": st.qkv, "act": st.act, "h": st.h}
    if c["op"] == "head":
        m, n, k = c["rows"], c["vocab"], c["hidden"]
        hip.rmsnorm(st.norm, st.h, st.nw, m, k, EPS)
        if c["logits"]:
            gemm = hip.gemm_small_w4a16 if c["bits"] == 4 else hip.gemm_small_w8a16
            gemm(st.logits, st.w, st.norm, m, st.scratch)
            hip.argmax_rows(st.idx, st.logits, m, n)
            return {"logits": st.logits, "idx": st.idx}
        greedy = hip.gemv_argmax_w4a16 if c["bits"] == 4 else hip.gemv_argmax_w8a16
        greedy(st.idx, st.w, st.norm, m, st.scratch)
        return {"norm": st.norm, "idx": st.idx}
    row = 0
    for (packed, scale, zp), n in zip(st.parts, _parts(c)):
        hip.awq_repack_into(st.w, row, packed, scale, zp, n)
        row += n
    hip.w4a16_dequant_rows(st.rows, st.w, 0, row)
    return st.rows


# -------------------------------------------------------------------- work
def _int4_bytes(n, k):
    return n * k // 2 + n * (k // GROUP) * 5 // 2   # levels, bf16 scales, 4-bit zero points


def work(case):
    c = case
    if c["op"] == "call":
        n, k = c["n"], c["k"]
        return {"bytes": _int4_bytes(n, k) + 2 * k + (4 if c["f32"] else 2) * n, "flops": 2 * n * k}
    if c["op"] == "layers":
        m, h, a, i = c["rows"], c["hidden"], c["attn"], c["inter"]
        mats = ((c["qkv"], h), (h, a), (2 * i, h), (h, i))
        w = sum(_int4_bytes(n, k) for n, k in mats)
        per = w + 4 * h + 2 * m * (a + c["qkv"])
        return {"bytes": c["layers"] * per + 2 * m * (2 * h + i),
                "flops": c["layers"] * 2 * m * sum(n * k for n, k in mats)}
    if c["op"] == "head":
        n, k, m = c["vocab"], c["hidden"], c["rows"]
        w = _int4_bytes(n, k) if c["bits"] == 4 else n * k + 2 * n * (k // GROUP)
        return {"bytes": w + 2 * m * k + 2 * k + (2 * m * n if c["logits"] else 2 * m * k) + 4 * m,
                "flops": 2 * m * n * k}
    n, k = sum(_parts(c)), c["k"]
    return {"bytes": 2 * _int4_bytes(n, k) + 2 * n * k, "flops": 0}


def tolerance(case):
    """Outputs are bf16 (2^-9 per rounding), or fp32 sums of a bare call. Two
    correct implementations round the same sums differently now and then, and a
    flipped rounding of one step travels through the steps after it. Figures:
    about four times the distance from exact()."""
    if case["op"] == "load":
        return "exact"
    if case["op"] == "call" and case["f32"]:
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 0.01, "max": 0.1}


# ------------------------------------------------------------------- exact
def _deq64(src):
    """[n][k] float64 of one compressed-tensors source."""
    packed, scale, zp = src
    n, words = packed.shape
    sh = torch.arange(0, 32, 4, device=packed.device, dtype=torch.int32)
    q = ((packed.unsqueeze(-1) >> sh) & 15).reshape(n, words * 8)
    z = ((zp.unsqueeze(1) >> sh.view(1, 8, 1)) & 15).reshape(n, -1)   # row 8 i + e of word i
    w = (q.view(n, -1, GROUP) - z.unsqueeze(-1)).to(torch.float64) * scale.to(torch.float64).unsqueeze(-1)
    return w.reshape(n, words * 8)


def _norm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * (1.0 + w.double())


def exact(case, seed):
    c = case
    g = _gen(seed)
    if c["op"] == "call":
        w = _deq64(_int4(g, c["n"], c["k"]))
        return _hidden(g, 1, c["k"]).double() @ w.T
    if c["op"] == "layers":
        table, ids = _embedding(g, c)
        h = table[ids].double()
        qkv, act = [], None
        for _ in range(c["layers"]):
            x = _layer_inputs(g, c, _int4)
            qkv.append(_norm64(h, x["n1"]) @ _deq64(x["qkv"]).T)
            h = h + x["attn"].double() @ _deq64(x["o"]).T
            gate, up = (_norm64(h, x["n2"]) @ _deq64(x["gu"]).T).split(c["inter"], -1)
            act = torch.nn.functional.silu(gate) * up
            h = h + act @ _deq64(x["down"]).T
        return {"qkv": qkv, "act": act, "h": h}
    if c["op"] == "head":
        n, k, m = c["vocab"], c["hidden"], c["rows"]
        x = _norm64(_hidden(g, m, k).double(), 0.1 * _bf16(g, k))
        if not c["logits"]:
            return {"norm": x, "idx": None}
        out = torch.empty(m, n, dtype=torch.float64, device="cuda")
        if c["bits"] == 4:
            packed, scale, zp = _int4(g, n, k)
        else:
            rows = _head_rows(g, n, k)
        for a in range(0, n, 8192):
            b = min(n, a + 8192)
            if c["bits"] == 4:
                w = _deq64((packed[a:b], scale[a:b], zp[a // 8:b // 8]))
            else:
                f = rows[a:b].float().view(b - a, -1, GROUP)
                top = f.abs().amax(-1, keepdim=True)
                q = (f * (127.0 / top)).round().clamp(-127, 127)
                w = (q.double() * (top / 127.0).to(torch.bfloat16).double()).view(b - a, k)
            out[:, a:b] = x @ w.T
        return {"logits": out, "idx": None}
    rows = [_deq64(_int4(g, n, c["k"])) for n in _parts(c)]
    return torch.cat(rows).to(torch.bfloat16).double()
