"""The calls whose speed this framework answers for, with the sizes they are made at.

Each case is one call a program makes through the C ABI (include/q8gemv.h,
include/qwen3_decode.h) on device memory it owns, at the shapes of
Qwen3-0.6B, the model the kernels are built for.  Weights, activations and
cache rows are drawn on the device from the seed, with the distributions of the
package's own synthetic model (matrices N(0, 0.02) quantized to Q8_0, norm
weights 1 + N(0, 0.1), embedding and output matrix N(0, 0.02)).

  listed()       the named cases
  draw(rng)      one more case of the same ranges
  prepare        what the program holds before the call
  run            the call, and what it wrote
  work           bytes and operations the call cannot do without
  tolerance      how far another correct implementation may be off
  exact          the same results in 64 bits, in plain torch
"""
from __future__ import annotations

import ctypes
import importlib.util
import math
import sys
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parent.parent / "qwen3-iree_amd"


def _package():
    name = "qwen3_iree_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            name, _PKG / "__init__.py", submodule_search_locations=[str(_PKG)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    import qwen3_iree_amd.decode as decode
    import qwen3_iree_amd.q8gemv as q8gemv
    return q8gemv, decode


Q, D = _package()

LAYERS, HIDDEN, FFN, VOCAB = 28, 1024, 3072, 151936
Q_DIM, KV_DIM, HEAD = 2048, 1024, 128
EPS, ROPE_BASE = 9.99999997e-7, 1.0e6
# rows and columns of a layer's Q8_0 matrices
SHAPES = {"wq": (Q_DIM, HIDDEN), "wk": (KV_DIM, HIDDEN), "wv": (KV_DIM, HIDDEN),
          "wo": (HIDDEN, Q_DIM), "wgu": (2 * FFN, HIDDEN), "wdn": (HIDDEN, FFN)}
SWEEP = ("wq", "wk", "wo", "wgu", "wdn")  # one matrix of each of the five kinds
LAYER_WEIGHTS = sum(n * k for n, k in SHAPES.values())
LAYER_Q8 = LAYER_WEIGHTS // 32 * 34


# ------------------------------------------------------------------ cases ----

def listed():
    return [
        # The six substituted dispatches of one layer, each its own call in the
        # layer's order: the smallest calls, as a runtime that replaces the
        # reference's executables one by one makes them.
        {"name": "layer_dispatches", "op": "dispatches", "layers": 1, "fused_qkv": False},
        # Every Q8_0 GEMV of the model (28 layers) in one batched launch: the
        # headline sweep.
        {"name": "sweep_28_layers", "op": "sweep", "layers": 28, "cut": 0},
        # Logits and token over the whole vocabulary.
        {"name": "vocab_argmax", "op": "vocab", "rows": VOCAB},
        # One layer of a decode step as its own call, at a chat-sized context.
        {"name": "decode_layer_ctx300", "op": "decode_layer", "ctx": 300},
        # A whole decode step: the context of the bench, and a long one.
        {"name": "decode_step_ctx1024", "op": "decode_step", "ctx": 1024},
        {"name": "decode_step_ctx16384", "op": "decode_step", "ctx": 16384},
        # One layer of prompt ingestion: a short chat turn; a turn on top of a
        # longer conversation, over the Q8_0 weights alone (no f16 copies kept);
        # a page of text; a long document.
        {"name": "prompt_layer_n33", "op": "prompt_layer", "n": 33, "start": 0, "f16": True,
         "chunk_local": False},
        {"name": "prompt_layer_q8_n300_at1700", "op": "prompt_layer", "n": 300, "start": 1700,
         "f16": False, "chunk_local": False},
        {"name": "prompt_layer_n512", "op": "prompt_layer", "n": 512, "start": 0, "f16": True,
         "chunk_local": False},
        {"name": "prompt_layer_n2048", "op": "prompt_layer", "n": 2048, "start": 0, "f16": True,
         "chunk_local": False},
        # (Whole steps and prompts answer with their logits and cache rows; the
        # token is those logits' argmax, which a last-bit difference can move
        # between two near-equal ones.  vocab_argmax answers with the token.)
        # Whole prompts: the chat-sized one of the bench's generation run, and a
        # ragged longer one.
        {"name": "prompt_n24", "op": "prompt", "n": 24, "f16": True},
        {"name": "prompt_n1021", "op": "prompt", "n": 1021, "f16": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["dispatches", "sweep", "vocab", "decode_layer", "decode_step", "prompt_layer",
                     "prompt_layer", "prompt_layer", "prompt"])
    if op == "dispatches":
        return {"op": op, "layers": rng.randint(1, 28), "fused_qkv": rng.random() < 0.5}
    if op == "sweep":
        return {"op": op, "layers": rng.randint(1, 28), "cut": rng.randint(0, 63)}
    if op == "vocab":
        return {"op": op, "rows": _log(rng, 1000, VOCAB)}
    if op in ("decode_layer", "decode_step"):
        return {"op": op, "ctx": _log(rng, 1, 16384)}
    if op == "prompt_layer":
        return {"op": op, "n": _log(rng, 1, 3000), "start": rng.choice([0, _log(rng, 1, 6000)]),
                "f16": rng.random() < 0.75, "chunk_local": rng.random() < 0.25}
    return {"op": op, "n": _log(rng, 1, 1021), "f16": rng.random() < 0.75}


# ----------------------------------------------------------------- inputs ----

def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(seed * 7919 + 17)
    return g


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.float16):
    out = torch.empty(shape, dtype=torch.float32, device="cuda")
    return out.normal_(mean, std, generator=g).to(dtype)


def _q8(g, rows, cols):
    """[rows, cols / 32, 34] bytes: Q8_0 blocks (f16 scale, 32 int8) of N(0, 0.02) values."""
    w = _normal(g, (rows * cols // 32, 32), 0.02, dtype=torch.float32)
    d = (w.abs().amax(1, keepdim=True) / 127.0).half()
    q = torch.round(w / d.float()).clamp_(-127, 127).to(torch.int8)
    out = torch.empty((rows, cols // 32, 34), dtype=torch.uint8, device="cuda")
    flat = out.view(-1, 34)
    flat[:, :2] = d.view(torch.uint8)
    flat[:, 2:] = q.view(torch.uint8)
    return out


def _q8_stack(g, name, layers):
    n, k = SHAPES[name]
    out = torch.empty((layers, n, k // 32, 34), dtype=torch.uint8, device="cuda")
    for i in range(layers):
        out[i] = _q8(g, n, k)
    return out


def _layer_params(g, layers):
    p = {name: _q8_stack(g, name, layers) for name in SHAPES}
    p["attn_norm"] = _normal(g, (layers, HIDDEN), 0.1, 1.0)
    p["ffn_norm"] = _normal(g, (layers, HIDDEN), 0.1, 1.0)
    p["q_norm"] = _normal(g, (layers, HEAD), 0.1, 1.0)
    p["k_norm"] = _normal(g, (layers, HEAD), 0.1, 1.0)
    return p


def _model_params(g, layers, vocab):
    """`layers` layers, with the embedding and output matrices if `vocab`."""
    p = _layer_params(g, layers)
    if vocab:
        p["token_embd"] = _normal(g, (VOCAB, HIDDEN), 0.02)
        p["output_norm"] = _normal(g, (HIDDEN,), 0.1, 1.0)
        p["output_w"] = _normal(g, (VOCAB, HIDDEN), 0.02)
    else:  # not read by a layer's call
        p["token_embd"] = p["output_norm"] = p["output_w"] = p["attn_norm"]
    return p


def _caches(g, layers, max_seq, filled):
    """K rows like normed, rotated heads; V rows like projections; `filled` slots in use."""
    k = torch.zeros((layers, max_seq, KV_DIM), dtype=torch.float16, device="cuda")
    v = torch.zeros((layers, max_seq, KV_DIM), dtype=torch.float16, device="cuda")
    for i in range(layers if filled else 0):
        k[i, :filled] = _normal(g, (filled, KV_DIM))
        v[i, :filled] = _normal(g, (filled, KV_DIM), 0.6)
    return k, v


def _inputs(case, seed):
    """The tensors a case starts from, made from the seed alone."""
    g = _gen(seed)
    op, t = case["op"], {}
    if op in ("dispatches", "sweep"):
        for name in SHAPES:
            t[name] = _q8_stack(g, name, case["layers"])
        for k in (1024, 2048, 3072):
            t["x%d" % k] = _normal(g, (k,))
    elif op == "vocab":
        t["w"] = _normal(g, (case["rows"], HIDDEN), 0.02)
        t["x"] = _normal(g, (HIDDEN,))
    elif op == "decode_layer":
        t["params"] = _model_params(g, 1, False)
        t["k"], t["v"] = _caches(g, 1, case["ctx"], case["ctx"] - 1)
        t["h"] = _normal(g, (HIDDEN,), 0.5)
    elif op == "decode_step":
        t["params"] = _model_params(g, LAYERS, True)
        t["k"], t["v"] = _caches(g, LAYERS, case["ctx"], case["ctx"] - 1)
        t["token"] = int(torch.randint(VOCAB, (1,), generator=_gen(seed, "cpu")))
    elif op == "prompt_layer":
        t["params"] = _model_params(g, 1, False)
        t["k"], t["v"] = _caches(g, 1, case["start"] + case["n"], case["start"])
        t["h"] = _normal(g, (case["n"], HIDDEN), 0.5)
    elif op == "prompt":
        t["params"] = _model_params(g, LAYERS, True)
        t["k"], t["v"] = _caches(g, LAYERS, case["n"], 0)
        t["prompt"] = torch.randint(VOCAB, (case["n"],), generator=_gen(seed, "cpu"))
    else:
        raise ValueError(op)
    return t


# ------------------------------------------------------------- the program ----

def _weights(p, f16_layers=0):
    """struct qwen3_weights over the tensors in `p`."""
    w = D.WeightsC(*(p[f].data_ptr() for f in D.WEIGHT_FIELDS), None)
    if not f16_layers:
        return w, None
    lib = Q.load_library()
    nbytes = lib.qwen3_prefill_matrices_bytes()
    if f16_layers < LAYERS:  # the expansion walks whole stacks: repeat the layer's
        full = dict(p, **{n: p[n].expand(LAYERS, *p[n].shape[1:]).contiguous() for n in SHAPES})
        src = D.WeightsC(*(full[f].data_ptr() for f in D.WEIGHT_FIELDS), None)
    else:
        full, src = p, w
    m = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    Q.check(lib.qwen3_prefill_matrices_expand(ctypes.byref(src), m.data_ptr(), nbytes, _stream()),
            "qwen3_prefill_matrices_expand")
    torch.cuda.synchronize()
    m = m[:nbytes // LAYERS * f16_layers].clone() if f16_layers < LAYERS else m
    w.prefill_f16 = m.data_ptr()
    return w, m


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _zeros(*shape, dtype=torch.float16):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    Q.init()
    lib = Q.load_library()
    s = _inputs(case, seed)
    s["op"], s["stream"] = case["op"], _stream()
    op = case["op"]
    if op == "dispatches":
        y = s["y"] = {n: _zeros(case["layers"], SHAPES[n][0]) for n in SHAPES}
        x = {k: s["x%d" % k].data_ptr() for k in (1024, 2048, 3072)}
        w = {n: s[n].data_ptr() for n in SHAPES}
        calls = s["calls"] = []
        for l in range(case["layers"]):
            at = {n: y[n][l].data_ptr() for n in SHAPES}
            if case["fused_qkv"]:
                calls.append((Q.q8gemv_qkv, (w["wq"], w["wk"], w["wv"], l, x[1024], at["wq"],
                                             at["wk"], at["wv"], s["stream"])))
            else:
                calls += [(Q.q8gemv, (kind, w[n], l, x[1024], at[n], s["stream"]))
                          for n, kind in (("wq", 0), ("wk", 1), ("wv", 1))]
            calls += [(Q.q8gemv, (kind, w[n], l, x[k], at[n], s["stream"]))
                      for n, kind, k in (("wo", 2, 2048), ("wgu", 3, 1024), ("wdn", 4, 3072))]
    elif op == "sweep":
        y = s["y"] = {n: _zeros(case["layers"], SHAPES[n][0] - case["cut"]) for n in SWEEP}
        s["batch"] = Q.Q8Batch([
            Q.desc(s[n][l].data_ptr(), SHAPES[n][0] - case["cut"], SHAPES[n][1],
                   s["x%d" % SHAPES[n][1]].data_ptr(), y[n][l].data_ptr())
            for l in range(case["layers"]) for n in SWEEP])
    elif op == "vocab":
        s["logits"] = _zeros(case["rows"])
        s["tok"] = _zeros(1, dtype=torch.int32)
        s["ws"] = _zeros(Q.vocab_workspace_bytes(), dtype=torch.uint8)
    elif op in ("decode_layer", "decode_step"):
        s["w"], _ = _weights(s["params"])
        s["scratch"] = _zeros(lib.qwen3_scratch_bytes(), dtype=torch.uint8)
        Q.check(lib.qwen3_scratch_reset(s["scratch"].data_ptr(), s["stream"]), "scratch_reset")
        pos = case["ctx"] - 1
        s["state"] = torch.tensor([s.get("token", 0), pos], dtype=torch.int32, device="cuda")
        s["first"] = s["state"].clone()
        s["h_out"] = _zeros(HIDDEN)
        s["logits"] = _zeros(VOCAB) if op == "decode_step" else None
        s["k_new"], s["v_new"] = s["k"][:, pos], s["v"][:, pos]
    else:
        layers = 1 if op == "prompt_layer" else LAYERS
        s["w"], s["f16"] = _weights(s["params"], layers if case["f16"] else 0)
        n = case["n"]
        s["ws_bytes"] = lib.qwen3_prefill_workspace_bytes(n)
        s["ws"] = _zeros(s["ws_bytes"], dtype=torch.uint8)
        if op == "prompt_layer":
            at = lib.qwen3_prefill_workspace_offset(n, b"h")
            s["h_io"] = s["ws"][at:at + n * HIDDEN * 2].view(torch.float16).view(n, HIDDEN)
            s["n"], s["start"], s["local"] = n, case["start"], int(case["chunk_local"])
            s["k_new"], s["v_new"] = s["k"][:, case["start"]:], s["v"][:, case["start"]:]
        else:
            s["prompt"] = s["prompt"].to(torch.int32).cuda()
            s["n"] = n
            s["scratch"] = _zeros(lib.qwen3_scratch_bytes(), dtype=torch.uint8)
            Q.check(lib.qwen3_scratch_reset(s["scratch"].data_ptr(), s["stream"]), "scratch_reset")
            s["state"] = _zeros(2, dtype=torch.int32)
            s["first"] = s["state"].clone()
            s["logits"] = _zeros(VOCAB)
    return s


def run(s):
    lib, op, st = Q.load_library(), s["op"], s["stream"]
    if op == "dispatches":
        for fn, args in s["calls"]:
            fn(*args)
        return s["y"]
    if op == "sweep":
        s["batch"].launch(st)
        return s["y"]
    if op == "vocab":
        Q.f16_gemv_argmax_rows(s["w"].data_ptr(), s["w"].shape[0], s["x"].data_ptr(),
                               s["logits"].data_ptr(), s["tok"].data_ptr(), s["ws"].data_ptr(), st)
        return {"logits": s["logits"], "token": s["tok"]}
    if op == "decode_layer":
        Q.check(lib.qwen3_decode_layer(
            ctypes.byref(s["w"]), 0, s["k"].data_ptr(), s["v"].data_ptr(), s["k"].shape[1],
            s["state"].data_ptr() + 4, s["h"].data_ptr(), s["h_out"].data_ptr(),
            s["scratch"].data_ptr(), st), "qwen3_decode_layer")
        return {"h": s["h_out"], "k": s["k_new"], "v": s["v_new"]}
    if op == "decode_step":
        s["state"].copy_(s["first"])  # the program's choice of token and position
        Q.check(lib.qwen3_decode_step(
            ctypes.byref(s["w"]), s["k"].data_ptr(), s["v"].data_ptr(), s["k"].shape[1],
            s["state"].data_ptr(), s["state"].data_ptr() + 4, s["logits"].data_ptr(), 0,
            s["scratch"].data_ptr(), st), "qwen3_decode_step")
        return {"logits": s["logits"], "k": s["k_new"], "v": s["v_new"]}
    if op == "prompt_layer":
        s["h_io"].copy_(s["h"])  # the layer's input rows, replaced by its output
        Q.check(lib.qwen3_prefill_layer(
            ctypes.byref(s["w"]), 0, s["k"].data_ptr(), s["v"].data_ptr(), s["k"].shape[1],
            s["n"], s["start"], s["local"], s["ws"].data_ptr(), s["ws_bytes"], st),
            "qwen3_prefill_layer")
        return {"h": s["h_io"], "k": s["k_new"], "v": s["v_new"]}
    s["state"].copy_(s["first"])
    Q.check(lib.qwen3_prefill_batched(
        ctypes.byref(s["w"]), s["k"].data_ptr(), s["v"].data_ptr(), s["k"].shape[1],
        s["prompt"].data_ptr(), s["n"], s["state"].data_ptr(), s["state"].data_ptr() + 4,
        s["logits"].data_ptr(), 0, s["ws"].data_ptr(), s["ws_bytes"], s["scratch"].data_ptr(), st),
        "qwen3_prefill_batched")
    return {"logits": s["logits"], "k": s["k"], "v": s["v"]}


# ------------------------------------------------------------ what it costs ----

def _attended(n, start, local):
    """(query, position) pairs of n tokens at `start`."""
    return n * (n + 1) // 2 + (0 if local else n * start)


def work(case):
    op = case["op"]
    if op == "dispatches":
        outs = sum(n for n, _ in SHAPES.values())
        return {"bytes": case["layers"] * (LAYER_Q8 + 2 * outs) + 2 * (1024 + 2048 + 3072),
                "flops": 2 * LAYER_WEIGHTS * case["layers"]}
    if op == "sweep":
        rows = [(SHAPES[n][0] - case["cut"], SHAPES[n][1]) for n in SWEEP]
        return {"bytes": case["layers"] * sum(r * k // 32 * 34 + 2 * r for r, k in rows) + 2 * 6144,
                "flops": 2 * case["layers"] * sum(r * k for r, k in rows)}
    if op == "vocab":
        return {"bytes": case["rows"] * (2 * HIDDEN + 2) + 2 * HIDDEN + 4,
                "flops": 2 * HIDDEN * case["rows"]}
    if op in ("decode_layer", "decode_step"):
        layers = 1 if op == "decode_layer" else LAYERS
        head = VOCAB * (2 * HIDDEN + 2) if op == "decode_step" else 0
        return {"bytes": layers * (LAYER_Q8 + 2 * 2 * KV_DIM * case["ctx"]) + head + 4 * HIDDEN,
                "flops": layers * (2 * LAYER_WEIGHTS + 4 * Q_DIM * case["ctx"]) + head}
    n, start, local = case["n"], case.get("start", 0), case.get("chunk_local", False)
    layers = 1 if op == "prompt_layer" else LAYERS
    head = VOCAB * (2 * HIDDEN + 2) if op == "prompt" else 0
    matrices = 2 * LAYER_WEIGHTS if case["f16"] else LAYER_Q8
    kv = 2 * 2 * KV_DIM * (n + (0 if local else start))
    return {"bytes": layers * (matrices + kv) + 2 * 2 * HIDDEN * n + head,
            "flops": layers * (2 * LAYER_WEIGHTS * n + 4 * Q_DIM * _attended(n, start, local)) + head}


def tolerance(case):
    """About four times the error measured against exact(): single GEMVs round
    once to f16 (2.1e-4), a layer's f16 chain shows 3e-4 to 5.6e-4, 28 layers 1.6e-3
    to 2.1e-3 for prompts and 2.9e-3 to 5.4e-3 for a step over a drawn cache."""
    return {"rel": {"dispatches": 8e-4, "sweep": 8e-4, "vocab": 8e-4, "decode_layer": 2e-3,
                    "prompt_layer": 2e-3, "prompt": 8e-3, "decode_step": 2e-2}[case["op"]]}


# --------------------------------------------------------- the same in 64 bits ----

def _f64(blocks):
    """[rows, cols / 32, 34] Q8_0 bytes -> f64 [rows, cols]."""
    d = blocks[..., :2].contiguous().view(torch.float16).double()
    q = blocks[..., 2:].contiguous().view(torch.int8).double()
    return (d * q).reshape(blocks.shape[0], -1)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    """x [tokens, heads, 128] at positions pos [tokens]."""
    i = torch.arange(HEAD // 2, device=x.device, dtype=torch.float64)
    th = pos.double()[:, None] * ROPE_BASE ** (-2.0 * i / HEAD)
    c, s = torch.cos(th)[:, None], torch.sin(th)[:, None]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _layer(p, l, h, k_old, v_old, start):
    """Layer l of h [n, 1024] at positions start..; k_old, v_old [m, 1024] the
    rows it also attends to.  Returns the output and the new K and V rows."""
    n, m = h.shape[0], k_old.shape[0]
    w = {name: _f64(p[name][l]) for name in SHAPES}
    pos = torch.arange(start, start + n, device=h.device)
    x = _norm(h, p["attn_norm"][l])
    q = _rope(_norm((x @ w["wq"].T).view(n, 16, HEAD), p["q_norm"][l]), pos)
    k = _rope(_norm((x @ w["wk"].T).view(n, 8, HEAD), p["k_norm"][l]), pos)
    v = (x @ w["wv"].T).view(n, 8, HEAD)
    keys = torch.cat([k_old.double().view(m, 8, HEAD), k])
    vals = torch.cat([v_old.double().view(m, 8, HEAD), v])
    out = torch.empty_like(q)
    for a in range(0, n, 512):
        b = min(n, a + 512)
        seen = torch.arange(m + n, device=h.device)[None] <= m + torch.arange(a, b, device=h.device)[:, None]
        for i in range(16):
            s = q[a:b, i] @ keys[:, i // 2].T / math.sqrt(HEAD)
            out[a:b, i] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ vals[:, i // 2]
    res = h + out.reshape(n, Q_DIM) @ w["wo"].T
    gu = _norm(res, p["ffn_norm"][l]) @ w["wgu"].T
    gate, up = gu[:, :FFN], gu[:, FFN:]
    return (res + (gate * torch.sigmoid(gate) * up) @ w["wdn"].T, k.reshape(n, KV_DIM),
            v.reshape(n, KV_DIM))


def exact(case, seed):
    t, op = _inputs(case, seed), case["op"]
    if op == "dispatches":
        return {n: torch.stack([_f64(w) @ t["x%d" % SHAPES[n][1]].double() for w in t[n]])
                for n in SHAPES}
    if op == "sweep":
        return {n: torch.stack([_f64(w)[:SHAPES[n][0] - case["cut"]] @
                                t["x%d" % SHAPES[n][1]].double() for w in t[n]]) for n in SWEEP}
    if op == "vocab":
        return {"logits": t["w"].double() @ t["x"].double(), "token": None}
    p = t["params"]
    if op in ("decode_layer", "prompt_layer"):
        prompt = op == "prompt_layer"
        start = case["start"] if prompt else case["ctx"] - 1
        h = t["h"].double().view(-1, HIDDEN)
        old = 0 if prompt and case["chunk_local"] else start
        h, k, v = _layer(p, 0, h, t["k"][0, :old], t["v"][0, :old], start)
        if not prompt:
            h = h[0]
        return {"h": h, "k": k.view(1, *k.shape) if prompt else k, "v": v.view(1, *v.shape) if prompt else v}
    step = op == "decode_step"
    start = case["ctx"] - 1 if step else 0
    ids = torch.tensor([t["token"]]) if step else t["prompt"]
    h = p["token_embd"][ids.cuda()].double()
    ks, vs = [], []
    for l in range(LAYERS):
        h, k, v = _layer(p, l, h, t["k"][l, :start], t["v"][l, :start], start)
        ks.append(k[0] if step else k)
        vs.append(v[0] if step else v)
    logits = p["output_w"].double() @ _norm(h[-1], p["output_norm"])
    return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}
