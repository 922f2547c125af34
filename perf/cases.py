"""Performance cases: the work a user of the backend has it do, through the
public entry points of hymt2sharp_amd.HipBackend.

Five kinds of case:

attn_decode   attention of one token at position `pos` through `layers`
              layers (decode_dev), call by call or as one recorded step
              (graph_launch), for each cache type;
attn_prefill  causal attention of `seq` prompt rows over `pos` cached
              positions, one layer (prefill_dev);
layers        what a layer does outside attention, for `rows` tokens: RMSNorm,
              the q/k/v projection, the o projection onto the residual,
              RMSNorm, gate/up, SwiGLU, the down projection onto the residual.
              One row is a decode step's chain of GEMVs (recorded), several
              rows are a prompt's GEMMs;
lm_head       the output norm and the output projection of one token;
turn          a turn of a conversation or a text to translate: ForwardStep over
              the prompt, then ForwardStep for each of the next tokens.

The shapes are the 32-layer model's: hidden 2048, FFN 6144, 16 q / 4 kv heads
of 128, vocabulary 120818.  Weights are Q4_K with a Q6_K embedding, as in the
Q4_K_M files, or another supported type; caches bf16 (the model's default),
fp16 or fp32.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from hymt2sharp_amd import HipBackend
from hymt2sharp_amd import _native as N
from hymt2sharp_amd.model import ModelConfig, Tensor

HIDDEN, FFN, HEADS, KV_HEADS, DIM, VOCAB, LAYERS = 2048, 6144, 16, 4, 128, 120818, 32
QD, KD = HEADS * DIM, KV_HEADS * DIM
BASE, EPS = 10000.0, 1e-6
DTYPES = {"f32": (N.F32, 4), "f16": (N.F16, 2), "bf16": (N.BF16, 2)}
# GGUF bytes per weight of the types the cases use
WEIGHTS = {"q4_k": (N.W_Q4_K, 144 / 256), "q6_k": (N.W_Q6_K, 210 / 256), "q8_0": (N.W_Q8_0, 34 / 32),
           "f16": (N.W_F16, 2.0)}


def listed():
    return [
        # the shortest decode attention that is configured: a 512-position fp32
        # cache, one layer, called as a host calls it
        {"name": "attn_decode_512_f32", "kind": "attn_decode", "pos": 512, "cache": "f32", "layers": 1,
         "recorded": False, "peaked": False},
        # the decode step's attention at a 4k context, all 32 layers replayed
        # as one recorded step: the benchmark's headline configuration
        {"name": "attn_decode_4096_f16_x32", "kind": "attn_decode", "pos": 4096, "cache": "f16", "layers": LAYERS,
         "recorded": True, "peaked": False},
        # long-context decode with a few very large keys
        {"name": "attn_decode_32768_f16_x4", "kind": "attn_decode", "pos": 32768, "cache": "f16", "layers": 4,
         "recorded": False, "peaked": True},
        # a 2048-token prompt into an empty cache
        {"name": "attn_prefill_2048_bf16", "kind": "attn_prefill", "pos": 0, "seq": 2048, "cache": "bf16",
         "io": "bf16"},
        # a chunk appended to a long cache
        {"name": "attn_prefill_256_at_8192_f16", "kind": "attn_prefill", "pos": 8192, "seq": 256, "cache": "f16",
         "io": "f32"},
        # the last chunk of an 8192-token document, as the model chunks it
        {"name": "attn_prefill_2048_at_6144", "kind": "attn_prefill", "pos": 6144, "seq": 2048, "cache": "bf16",
         "io": "bf16"},
        # a decode step's GEMVs (8 layers, more than the last-level cache holds
        # of the rotating states)
        {"name": "layers_1_q4_k", "kind": "layers", "rows": 1, "weight": "q4_k", "layers": 8},
        # a sentence: the commonest prompt of a translation model
        {"name": "layers_61_q4_k", "kind": "layers", "rows": 61, "weight": "q4_k", "layers": 2},
        # a few paragraphs, a ragged length
        {"name": "layers_700_q4_k", "kind": "layers", "rows": 700, "weight": "q4_k", "layers": 2},
        # a full prefill chunk
        {"name": "layers_2048_q4_k", "kind": "layers", "rows": 2048, "weight": "q4_k", "layers": 2},
        # the output projection of every decode step and prompt
        {"name": "lm_head_q6_k", "kind": "lm_head", "rows": VOCAB, "weight": "q6_k"},
        # a short text translated by the whole model: the prompt, then the
        # first tokens of the answer
        {"name": "turn_301_plus_3", "kind": "turn", "tokens": 301, "next": 3},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn_decode", "attn_decode", "attn_prefill", "attn_prefill", "layers", "layers", "layers",
                       "lm_head", "turn"])
    if kind == "attn_decode":
        pos = _log_int(rng, 64, 32768)
        cache = rng.choice(["f32", "f16", "bf16"])
        return {"kind": kind, "pos": pos, "cache": cache, "layers": 1 if pos > 8192 else rng.choice([1, 4, 12]),
                "recorded": rng.random() < 0.5, "peaked": rng.random() < 0.3}
    if kind == "attn_prefill":
        return {"kind": kind, "pos": 0 if rng.random() < 0.5 else _log_int(rng, 64, 6144),
                "seq": _log_int(rng, 16, 2048), "cache": rng.choice(["f16", "bf16"]),
                "io": rng.choice(["f32", "bf16"])}
    if kind == "layers":
        return {"kind": kind, "rows": 1 if rng.random() < 0.2 else _log_int(rng, 2, 2048),
                "weight": rng.choice(["q4_k", "q4_k", "q6_k", "q8_0"]), "layers": 2}
    if kind == "lm_head":
        return {"kind": kind, "rows": _log_int(rng, 16384, VOCAB), "weight": rng.choice(["q6_k", "q4_k", "q8_0"])}
    return {"kind": kind, "tokens": _log_int(rng, 4, 300), "next": rng.choice([1, 2, 3])}


# ---- inputs ------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * scale


def _gamma(g, n):
    """A norm weight, U(0.9, 1.1)."""
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float32) * 0.2 + 0.9


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).view(-1, 2)


STD = 1.0 / math.sqrt(2048.0)  # a projection's weights: keeps values of order one


def _weight(g, name, rows, cols, std=STD):
    """rows x cols weights as rows of GGUF blocks (uint8 tensor on the GPU,
    [blocks][block bytes]): zero-mean values of standard deviation `std`."""

    def bytes_(*shape):
        return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)

    def u(n):
        return torch.rand(n, generator=g, device="cuda") * 0.5 + 0.75

    if name == "f16":
        return (_normal(g, rows, cols) * std).to(torch.float16).view(torch.uint8)
    if name == "q8_0":  # 32 values: fp16 d, int8
        nb = rows * cols // 32
        raw = torch.empty(nb, 34, dtype=torch.uint8, device="cuda")
        raw[:, 0:2] = _half_bytes(std / 73.9 * u(nb))
        raw[:, 2:] = bytes_(nb, 32)
        return raw
    nb = rows * cols // 256
    if name == "q6_k":  # 256 values: ql 128, qh 64, int8 scales 16, fp16 d
        raw = torch.empty(nb, 210, dtype=torch.uint8, device="cuda")
        raw[:, :192] = bytes_(nb, 192)
        raw[:, 192:208] = torch.randint(32, 96, (nb, 16), generator=g, device="cuda", dtype=torch.uint8)
        raw[:, 208:210] = _half_bytes(std / (18.5 * 64) * u(nb))
        return raw
    # q4_k, 256 values: fp16 d, dmin, 12 bytes of 6-bit scales and mins, 128
    # nibble bytes; min = 7.5 d scale makes a sub-block's values zero-mean
    sc = torch.randint(24, 64, (nb, 8), generator=g, device="cuda", dtype=torch.uint8)
    lo, hi = sc[:, :4], sc[:, 4:]
    d = std / (4.61 * 44) * u(nb)
    raw = torch.empty(nb, 144, dtype=torch.uint8, device="cuda")
    raw[:, 0:2] = _half_bytes(d)
    raw[:, 2:4] = _half_bytes(7.5 * d)
    raw[:, 4:8] = lo | ((hi >> 4) << 6)
    raw[:, 8:12] = lo | ((hi >> 4) << 6)
    raw[:, 12:16] = (hi & 15) | ((hi & 15) << 4)
    raw[:, 16:] = bytes_(nb, 128)
    return raw


def _host(t):
    return t.cpu().numpy().tobytes()


def _bf16_bits(t):
    return t.to(torch.bfloat16).view(torch.int16).cpu().numpy().view(np.uint16)


def _cached(g, n, peaked):
    """n cached rows of K (normalised: unit mean square; peaked: one position
    in a thousand 30 times larger) and V, as UploadKv takes them."""
    k, v = _normal(g, n, KD), _normal(g, n, KD)
    if peaked:
        at = torch.randint(0, n, (max(1, n // 1000),), generator=g, device="cuda")
        k[at] *= 30.0
    return k.to(torch.bfloat16), v.to(torch.bfloat16)


def _bits_in(cached):
    return tuple(t.view(torch.int16).cpu().numpy().view(np.uint16) for t in cached)


def _ptr(t):
    return t.data_ptr()


class _Room:
    """Layers of a shared KV cache, held while a state lives.  A program runs
    on one backend, whose calls follow each other on its stream; so the states
    of a case share a backend, each in cache layers of its own (they use the
    same positions, and the page table is one for all layers)."""

    STATES = 4
    shared = {"key": None, "rooms": []}

    def __init__(self, layers, max_tokens, cache):
        self.graph = None
        key, shared = (layers, max_tokens, cache), _Room.shared
        if shared["key"] != key or not shared["rooms"]:
            be = HipBackend(0).configure(HEADS, KV_HEADS, DIM, DIM, BASE, EPS)
            be.create_cache(layers * self.STATES, max_tokens, DTYPES[cache][0])
            shared["key"], shared["rooms"] = key, [(be, i * layers) for i in range(self.STATES)]
        self.key, self.rooms = key, shared["rooms"]
        self.be, self.first = self.rooms.pop(0)

    def __del__(self):
        try:
            if self.graph is not None:
                self.be.graph_destroy(self.graph)
            self.rooms.append((self.be, self.first))
        except Exception:  # the interpreter or the backend is going down
            pass


def _plain_backend():
    """The backend of the cases without a cache."""
    if _Room.shared.get("plain") is None:
        _Room.shared["plain"] = HipBackend(0)
    return _Room.shared["plain"]


class _Weights:
    """Uploaded weights, freed with the state that holds them."""

    def __init__(self, be):
        self.be, self.handles, self.graph = be, [], None

    def add(self, weight, raw, rows, cols, dense):
        h = self.be.weight_upload(WEIGHTS[weight][0], rows, cols, _host(raw))
        self.handles.append(h)
        if dense:
            self.be.weight_dense(h)
        return h

    def __del__(self):
        try:
            if self.graph is not None:
                self.be.graph_destroy(self.graph)
            for h in self.handles:
                self.be.weight_free(h)
        except Exception:  # the interpreter or the backend is going down
            pass


# ---- attention ---------------------------------------------------------------------


def _attn_decode_inputs(case, seed):
    g = _gen(seed)
    n = case["layers"]
    x = [(_normal(g, QD), _normal(g, KD), _normal(g, KD), _gamma(g, DIM), _gamma(g, DIM)) for _ in range(n)]
    return x, [_cached(g, case["pos"], case["peaked"]) for _ in range(n)]


def _prepare_attn_decode(case, seed):
    x, cached = _attn_decode_inputs(case, seed)
    room = _Room(case["layers"], case["pos"] + 64, case["cache"])
    be = room.be
    for l, c in enumerate(cached):
        be.UploadKv(room.first + l, 0, case["pos"], *_bits_in(c))
    out = torch.empty(case["layers"], QD, device="cuda")
    torch.cuda.synchronize()
    s = {"be": be, "room": room, "x": x, "out": out, "pos": case["pos"], "case": case}
    if case["recorded"]:
        _attn_decode_calls(s)
        be.sync()
        be.graph_begin()
        _attn_decode_calls(s)
        room.graph = be.graph_end()
    return s


def _attn_decode_calls(s):
    be, out, first = s["be"], s["out"], s["room"].first
    for l, (q, k, v, gq, gk) in enumerate(s["x"]):
        be.decode_dev(first + l, s["pos"], _ptr(q), _ptr(k), _ptr(v), _ptr(gq), _ptr(gk), _ptr(out[l]))


def _run_attn_decode(s):
    if s["room"].graph is not None:
        s["be"].graph_launch(s["room"].graph)
    else:
        _attn_decode_calls(s)
    return s["out"]


def _attn_prefill_inputs(case, seed):
    g = _gen(seed)
    S = case["seq"]
    q, k, v = _normal(g, S, QD), _normal(g, S, KD), _normal(g, S, KD)
    if case["io"] == "bf16":
        q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    return q, k, v, _gamma(g, DIM), _gamma(g, DIM), _cached(g, case["pos"], False) if case["pos"] else None


def _prepare_attn_prefill(case, seed):
    q, k, v, gq, gk, cached = _attn_prefill_inputs(case, seed)
    room = _Room(1, case["pos"] + case["seq"], case["cache"])
    if cached is not None:
        room.be.UploadKv(room.first, 0, case["pos"], *_bits_in(cached))
    out = torch.empty(case["seq"], QD, device="cuda")
    torch.cuda.synchronize()
    return {"be": room.be, "room": room, "x": (q, k, v, gq, gk), "out": out, "case": case}


def _run_attn_prefill(s):
    q, k, v, gq, gk = s["x"]
    c = s["case"]
    s["be"].prefill_dev(s["room"].first, c["pos"], c["seq"], _ptr(q), _ptr(k), _ptr(v), N.BF16 if c["io"] == "bf16" else N.F32,
                        _ptr(gq), _ptr(gk), _ptr(s["out"]))
    return s["out"]


# ---- the layer outside attention ---------------------------------------------------


def _layers_inputs(case, seed):
    g = _gen(seed)
    rows, wt = case["rows"], case["weight"]
    x0 = _normal(g, rows, HIDDEN)
    layers = []
    for _ in range(case["layers"]):
        layers.append({"attn_norm": _gamma(g, HIDDEN), "ffn_norm": _gamma(g, HIDDEN),
                       "ao": _normal(g, rows, QD),
                       "qkv": _weight(g, wt, QD + 2 * KD, HIDDEN), "o": _weight(g, wt, HIDDEN, QD),
                       "gate_up": _weight(g, wt, 2 * FFN, HIDDEN), "down": _weight(g, wt, HIDDEN, FFN)})
    return x0, layers


_SHAPES = {"qkv": (QD + 2 * KD, HIDDEN), "o": (HIDDEN, QD), "gate_up": (2 * FFN, HIDDEN), "down": (HIDDEN, FFN)}


def _prepare_layers(case, seed):
    x0, layers = _layers_inputs(case, seed)
    rows = case["rows"]
    be = _plain_backend()
    weights = _Weights(be)
    for L in layers:
        for name, (r, c) in _SHAPES.items():
            L[name] = weights.add(case["weight"], L[name], r, c, rows > 1)
    s = {"be": be, "x0": x0, "x": x0.clone(), "layers": layers, "weights": weights, "case": case,
         "stream": torch.cuda.ExternalStream(be.stream())}
    if rows == 1:
        s["qkv"] = torch.empty(len(layers), QD + 2 * KD, device="cuda")
        s["act"] = torch.empty(FFN, device="cuda")
        torch.cuda.synchronize()
        _decode_layer_calls(s)
        be.sync()
        be.graph_begin()
        _decode_layer_calls(s)
        weights.graph = be.graph_end()
        be.sync()
    else:
        h = dict(device="cuda", dtype=torch.bfloat16)
        s["xn"] = torch.empty(rows, HIDDEN, **h)
        s["qkv"] = torch.empty(len(layers), rows, QD + 2 * KD, **h)
        s["gu"] = torch.empty(rows, 2 * FFN, **h)
        s["act"] = torch.empty(rows, FFN, **h)
        for L in layers:  # the attention's output, rounded as the model hands it on
            L["ao"] = L["ao"].to(torch.bfloat16)
        torch.cuda.synchronize()
        # whether the fused gate/up + SwiGLU call serves this prompt length:
        # a program asks once
        try:
            be.gemm_swiglu(layers[0]["gate_up"], _ptr(s["xn"]), rows, _ptr(s["act"]))
            s["fused"] = True
        except N.NotSupportedError:
            s["fused"] = False
        be.sync()
    return s


def _decode_layer_calls(s):
    be, x = s["be"], _ptr(s["x"])
    for l, L in enumerate(s["layers"]):
        be.gemv(L["qkv"], x, _ptr(s["qkv"][l]), rmsnorm=_ptr(L["attn_norm"]), eps=EPS)
        be.gemv(L["o"], _ptr(L["ao"]), x, accumulate=True)
        be.gemv(L["gate_up"], x, _ptr(s["act"]), rmsnorm=_ptr(L["ffn_norm"]), eps=EPS, swiglu_out=True)
        be.gemv(L["down"], _ptr(s["act"]), x, accumulate=True)


def _run_layers(s):
    be, m = s["be"], s["case"]["rows"]
    with torch.cuda.stream(s["stream"]):  # the residual as the step before leaves it
        s["x"].copy_(s["x0"])
    if m == 1:
        be.graph_launch(s["weights"].graph)
        return [s["x"], s["qkv"]]
    x, xn, gu, act = (_ptr(s[n]) for n in ("x", "xn", "gu", "act"))
    for l, L in enumerate(s["layers"]):
        be.rows_rmsnorm(x, m, HIDDEN, _ptr(L["attn_norm"]), EPS, xn)
        be.gemm(L["qkv"], xn, m, _ptr(s["qkv"][l]), nrows=QD + 2 * KD, out_bf16=True)
        be.gemm(L["o"], _ptr(L["ao"]), m, x, nrows=HIDDEN, accumulate=True)
        be.rows_rmsnorm(x, m, HIDDEN, _ptr(L["ffn_norm"]), EPS, xn)
        if s["fused"]:
            be.gemm_swiglu(L["gate_up"], xn, m, act)
        else:
            be.gemm(L["gate_up"], xn, m, gu, nrows=2 * FFN, out_bf16=True)
            be.rows_swiglu_bf16(gu, m, FFN, act)
        be.gemm(L["down"], act, m, x, nrows=HIDDEN, accumulate=True)
    return [s["x"], s["qkv"]]


# ---- the output projection ---------------------------------------------------------


def _lm_head_inputs(case, seed):
    g = _gen(seed)
    return _normal(g, HIDDEN, scale=4.0), _gamma(g, HIDDEN), _weight(g, case["weight"], case["rows"], HIDDEN)


def _prepare_lm_head(case, seed):
    x, gamma, w = _lm_head_inputs(case, seed)
    be = _plain_backend()
    weights = _Weights(be)
    h = weights.add(case["weight"], w, case["rows"], HIDDEN, False)
    s = {"be": be, "weights": weights, "w": h, "x": x, "gamma": gamma, "y": torch.empty(case["rows"], device="cuda"), "case": case}
    torch.cuda.synchronize()
    return s


def _run_lm_head(s):
    s["be"].gemv(s["w"], _ptr(s["x"]), _ptr(s["y"]), rmsnorm=_ptr(s["gamma"]), eps=EPS)
    return s["y"]


# ---- the whole model ---------------------------------------------------------------


def _turn_layer(seed, l):
    """Layer l's norms and weight blocks, made from the seed alone."""
    g = _gen(seed * 1000 + 1 + l)
    t = {"attn_norm": _gamma(g, HIDDEN), "ffn_norm": _gamma(g, HIDDEN), "attn_q_norm": _gamma(g, DIM),
         "attn_k_norm": _gamma(g, DIM)}
    # what is added to the residual is scaled down with the depth, as training
    # starts from and as keeps one layer's share of the sum small
    add = STD / math.sqrt(2 * LAYERS)
    for name, r, c, std in (("attn_q", QD, HIDDEN, STD), ("attn_k", KD, HIDDEN, STD), ("attn_v", KD, HIDDEN, STD),
                            ("attn_output", HIDDEN, QD, add), ("ffn_gate", FFN, HIDDEN, STD),
                            ("ffn_up", FFN, HIDDEN, STD), ("ffn_down", HIDDEN, FFN, add)):
        t[name] = (_weight(g, "q4_k", r, c, std), r, c)
    return t


def _turn_inputs(case, seed):
    g = _gen(seed * 1000)
    embd, norm = _weight(g, "q6_k", VOCAB, HIDDEN, 1.0), _gamma(g, HIDDEN)
    ids = torch.randint(0, VOCAB, (case["tokens"] + case["next"],), generator=g, device="cuda")
    return embd, norm, ids.cpu().tolist()


def _prepare_turn(case, seed):
    embd, norm, ids = _turn_inputs(case, seed)

    def vec(t):
        return Tensor(N.W_F32, 1, t.numel(), _host(t))

    tensors = {"token_embd.weight": Tensor(N.W_Q6_K, VOCAB, HIDDEN, _host(embd)), "output_norm.weight": vec(norm)}
    for l in range(LAYERS):
        for name, t in _turn_layer(seed, l).items():
            tensors[f"blk.{l}.{name}.weight"] = Tensor(N.W_Q4_K, t[1], t[2], _host(t[0])) if isinstance(t, tuple) \
                else vec(t)
    be = HipBackend(0)
    be.LoadModel(tensors, ModelConfig(eps=EPS), max_tokens=1024)
    return {"be": be, "ids": ids, "case": case}


def _run_turn(s):
    be, ids, n = s["be"], s["ids"], s["case"]["tokens"]
    be.SetCacheLen(0)
    out = [be.ForwardStep(ids[:n], 0)]
    for i in range(n, len(ids)):
        out.append(be.ForwardStep(ids[i:i + 1], i))
    return out


def prepare(case, seed):
    return {"attn_decode": _prepare_attn_decode, "attn_prefill": _prepare_attn_prefill, "layers": _prepare_layers,
            "lm_head": _prepare_lm_head, "turn": _prepare_turn}[case["kind"]](case, seed)


def run(state):
    return {"attn_decode": _run_attn_decode, "attn_prefill": _run_attn_prefill, "layers": _run_layers,
            "lm_head": _run_lm_head, "turn": _run_turn}[state["case"]["kind"]](state)


# ---- what a pass cannot do without -------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "attn_decode":
        L, n, sz = case["pos"] + 1, case["layers"], DTYPES[case["cache"]][1]
        return {"bytes": n * (2 * L * KD * sz + QD * 8 + 2 * KD * 4 + 2 * DIM * 4), "flops": n * 4 * DIM * HEADS * L}
    if kind == "attn_prefill":
        P, S, sz = case["pos"], case["seq"], DTYPES[case["cache"]][1]
        io = 2 if case["io"] == "bf16" else 4
        return {"bytes": 2 * (P + S) * KD * sz + S * (QD * (io + 4) + 2 * KD * io),
                "flops": 4 * DIM * HEADS * (S * P + S * (S + 1) // 2)}
    if kind == "layers":
        m, n, bpw = case["rows"], case["layers"], WEIGHTS[case["weight"]][1]
        per = sum(r * c for r, c in _SHAPES.values())
        # several rows read the bf16 copies that weight_dense made
        wbytes = per * (bpw if m == 1 else 2)
        es = 4 if m == 1 else 2
        return {"bytes": n * (wbytes + m * (QD * es + (QD + 2 * KD) * es)) + 2 * m * HIDDEN * 4,
                "flops": n * 2 * m * per}
    if kind == "lm_head":
        w = case["rows"] * HIDDEN
        return {"bytes": w * WEIGHTS[case["weight"]][1] + 8 * HIDDEN + 4 * case["rows"], "flops": 2 * w}
    per = LAYERS * sum(r * c for r, c in _SHAPES.values())
    head, n, more = VOCAB * HIDDEN, case["tokens"], case["next"]
    att = 4 * DIM * HEADS * LAYERS * sum(range(1, n + more + 1))
    return {"bytes": per * (2 if n > 1 else 144 / 256) + more * per * 144 / 256
            + (1 + more) * (head * 210 / 256 + 4 * VOCAB)
            + LAYERS * 2 * KD * 2 * (n + sum(range(n + 1, n + more + 1))),
            "flops": 2 * per * (n + more) + 2 * head * (1 + more) + att}


def tolerance(case):
    """Largest relative error between two correct implementations at the same
    precision, about four times what was measured.  Decode attention and the
    GEMVs sum in fp32 (operands of the attention products split into two
    16-bit halves): 3e-7 to 3e-6 against 64 bits; a new K row on a rounding
    boundary may round the other way, a larger step in bf16.  A prompt's
    attention rounds q and the weights P to the cache type: 2.7e-3 (bf16) and
    3.6e-4 (f16) against 64 bits.  A prompt's GEMMs with their fp32 sums in
    another order differ by 7e-4 over two layers (bf16 roundings between
    them), 4e-3 in the logits after 32."""
    kind = case["kind"]
    if kind == "attn_decode":
        return {"rel": 1e-4, "max": 4e-3} if case["cache"] == "bf16" else {"rel": 2e-5, "max": 1e-3}
    if kind == "attn_prefill":
        return {"rel": 8e-3, "max": 0.1} if case["cache"] == "bf16" else {"rel": 1.5e-3, "max": 0.02}
    if kind == "layers":
        return {"rel": 1e-5, "max": 1e-4} if case["rows"] == 1 else {"rel": 3e-3, "max": 0.04}
    if kind == "lm_head":
        return {"rel": 5e-6, "max": 1e-4}
    return {"rel": 1.6e-2, "max": 0.08}


# ---- the same in 64 bits -----------------------------------------------------------


def _dequant(name, raw, rows, cols):
    """The blocks of _weight as fp64 [rows][cols]."""
    def half(b):
        return b.contiguous().view(torch.float16).double()

    if name == "f16":
        return raw.view(torch.float16).double().view(rows, cols)
    if name == "q8_0":
        return (half(raw[:, 0:2]) * raw[:, 2:].contiguous().view(torch.int8).double()).view(rows, cols)
    nb = raw.shape[0]
    if name == "q6_k":
        ql, qh = raw[:, :128].view(nb, 2, 2, 32), raw[:, 128:192].view(nb, 2, 32)
        # half h, quarter j of 32 values: the low nibbles of quarters 0, 1, then the high ones
        q = torch.stack([(ql[:, :, j & 1] >> (4 * (j >> 1))) & 15 | ((qh >> (2 * j)) & 3) << 4 for j in range(4)], 2)
        sc = raw[:, 192:208].contiguous().view(torch.int8).double().view(nb, 2, 4, 2, 1)
        v = (q.double() - 32).view(nb, 2, 4, 2, 16) * sc
        return (half(raw[:, 208:210]).view(nb, 1, 1, 1, 1) * v).view(rows, cols)
    s = raw[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
    qs = raw[:, 16:].view(nb, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).view(nb, 8, 32).double()
    d, dmin = half(raw[:, 0:2]).view(nb, 1, 1), half(raw[:, 2:4]).view(nb, 1, 1)
    return (d * sc.unsqueeze(2) * q - dmin * mn.unsqueeze(2)).view(rows, cols)


def _rms(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def _rope(x, pos):
    """Half-split rotation of x [n][heads][DIM] at positions pos..; the angle
    is the fp32 product that defines the rotation table."""
    half = DIM // 2
    i = torch.arange(half, device="cuda", dtype=torch.float32)
    freq = 1.0 / torch.pow(BASE, (i / half).double()).float()
    p = torch.arange(pos, pos + x.shape[0], device="cuda", dtype=torch.float32)
    a = (p[:, None] * freq[None, :]).double()[:, None, :]
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * a.cos() - hi * a.sin(), lo * a.sin() + hi * a.cos()], -1)


_STORE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _attend(q, k, v, gq, gk, kc, vc, pos, cache):
    """Attention of rows at positions pos.. over cached rows kc, vc [pos][KD]
    (None: none) and their own, which are rounded to the cache type.  Returns
    out [n][QD] and the K and V rows of the whole sequence."""
    n = q.shape[0]
    q = _rms(_rope(q.double().view(n, HEADS, DIM), pos), gq)
    k = _rms(_rope(k.double().view(n, KV_HEADS, DIM), pos), gk).to(_STORE[cache]).double()
    v = v.double().view(n, KV_HEADS, DIM).to(_STORE[cache]).double()
    if kc is not None:
        k, v = torch.cat([kc.view(pos, KV_HEADS, DIM), k]), torch.cat([vc.view(pos, KV_HEADS, DIM), v])
    out = torch.empty(n, HEADS, DIM, dtype=torch.float64, device="cuda")
    mask = torch.arange(pos + n, device="cuda")[None, :] > torch.arange(pos, pos + n, device="cuda")[:, None]
    for h in range(HEADS):
        kh, vh = k[:, h // 4], v[:, h // 4]
        s = (q[:, h] @ kh.t().contiguous()) / math.sqrt(DIM)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ vh.contiguous()
    return out.view(n, QD), k.reshape(-1, KD), v.reshape(-1, KD)


def _silu_mul(gu):
    g, u = gu[:, :FFN], gu[:, FFN:]
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn_decode":
        x, cached = _attn_decode_inputs(case, seed)
        return torch.cat([_attend(q[None], k[None], v[None], gq, gk, kc.double(), vc.double(), case["pos"],
                                  case["cache"])[0] for (q, k, v, gq, gk), (kc, vc) in zip(x, cached)])
    if kind == "attn_prefill":
        q, k, v, gq, gk, cached = _attn_prefill_inputs(case, seed)
        kc, vc = (None, None) if cached is None else (t.double() for t in cached)
        return _attend(q, k, v, gq, gk, kc, vc, case["pos"], case["cache"])[0]
    if kind == "layers":
        x0, layers = _layers_inputs(case, seed)
        x, qkv = x0.double(), []
        for L in layers:
            W = {name: _dequant(case["weight"], L[name], *_SHAPES[name]) for name in _SHAPES}
            ao = L["ao"] if case["rows"] == 1 else L["ao"].to(torch.bfloat16)
            qkv.append(_rms(x, L["attn_norm"]) @ W["qkv"].t())
            x = x + ao.double() @ W["o"].t()
            x = x + _silu_mul(_rms(x, L["ffn_norm"]) @ W["gate_up"].t()) @ W["down"].t()
        q = torch.stack(qkv)
        return [x, q.view(len(layers), -1) if case["rows"] == 1 else q]
    if kind == "lm_head":
        x, gamma, w = _lm_head_inputs(case, seed)
        xn = _rms(x.double()[None], gamma)
        per = HIDDEN * WEIGHTS[case["weight"]][1] / w.shape[1]  # blocks per row
        parts = [_dequant(case["weight"], w[int(r * per):int(min(case["rows"], r + 16384) * per)],
                          min(16384, case["rows"] - r), HIDDEN) @ xn[0] for r in range(0, case["rows"], 16384)]
        return torch.cat(parts)
    embd, norm, ids = _turn_inputs(case, seed)
    n = len(ids)
    blocks = embd.view(VOCAB, -1, 210)
    x = _dequant("q6_k", blocks[torch.tensor(ids, device="cuda")].reshape(-1, 210), n, HIDDEN)
    for l in range(LAYERS):
        t = _turn_layer(seed, l)
        W = {k: _dequant("q4_k", *v) for k, v in t.items() if isinstance(v, tuple)}
        xn = _rms(x, t["attn_norm"])
        q, k, v = (xn @ W[w].t() for w in ("attn_q", "attn_k", "attn_v"))
        ao = _attend(q, k, v, t["attn_q_norm"], t["attn_k_norm"], None, None, 0, "bf16")[0]
        x = x + ao @ W["attn_output"].t()
        xn = _rms(x, t["ffn_norm"])
        x = x + _silu_mul(torch.cat([xn @ W["ffn_gate"].t(), xn @ W["ffn_up"].t()], 1)) @ W["ffn_down"].t()
    last = _rms(x[case["tokens"] - 1:], norm)
    parts = [_dequant("q6_k", blocks[r:r + 16384].reshape(-1, 210), min(16384, VOCAB - r), HIDDEN) @ last.t()
             for r in range(0, VOCAB, 16384)]
    return list(torch.cat(parts).t().contiguous())
