"""The framework's work, as cases that can be timed and checked one by one.

Each case drives the C ABI (include/am_gfx950.h, include/am_runtime.h) the way a
program that serves a Llama-family model does: whole sessions, one decoder layer of a
decode step, one decoder layer of a prefill pass, decode attention over a long cache,
and the language-model head.  The layer cases run the calls the runtime's own plans
run, in the same order, with the weights, caches, tables and workspaces laid out once.
"""

from __future__ import annotations

import ctypes as C
import json
import math
import os
import struct
import tempfile

import numpy as np
import torch

import aethermind_amd.native as N

FORMATS = {"bf16": N.AM_WF_BF16, "int8": N.AM_WF_INT8, "int4": N.AM_WF_INT4}
GROUP = 128
EPS = 1e-5
THETA = 500000.0
EMBED_ROWS = 2048  # rows of the embedding table the layer cases gather from

# Layer shapes: the 8B shape of the benchmark and the 2048-wide one of the tests.
SHAPES = {
    "8b": {"hidden": 4096, "hq": 32, "hkv": 8, "d": 128, "ffn": 14336, "vocab": 128256},
    "2k": {"hidden": 2048, "hq": 16, "hkv": 4, "d": 128, "ffn": 5632, "vocab": 32000},
}
# The tiny fp32 configuration of the benchmark's first workload.
TINY = {"layers": 4, "hidden": 512, "hq": 8, "hkv": 2, "d": 64, "ffn": 1376, "vocab": 32000, "theta": 10000.0}


def listed():
    return [
        # A small fp32 model answering a short prompt from its checkpoint: the smallest
        # whole call, prefill and greedy decode through the session API.
        {"name": "generate_tiny_f32", "kind": "generate", "prompt": 48, "new": 32},
        # Time to first token of an ordinary prompt through the session API (two layers
        # of the 8B shape with the full vocabulary), logits read back.
        {"name": "session_prefill_int4_200", "kind": "session", "fmt": "int4", "layers": 2, "prompt": 200},
        # One layer of single-sequence decode, the headline workload: INT4, short context.
        {"name": "decode_int4_b1", "kind": "decode", "shape": "8b", "fmt": "int4", "rows": 1, "ctx": 640, "block": 0},
        # A few sequences decoded together on a paged cache, contexts of several lengths.
        {"name": "decode_int4_b4_paged", "kind": "decode", "shape": "8b", "fmt": "int4", "rows": 4, "ctx": 1100, "block": 64},
        # The widest batch a session decodes, INT8 weights, ragged contexts.
        {"name": "decode_int8_b16", "kind": "decode", "shape": "8b", "fmt": "int8", "rows": 16, "ctx": 777, "block": 0},
        # Long-context decode: attention over four 8k contexts (the benchmark's fifth workload).
        {"name": "attention_b4_8k", "kind": "attention", "rows": 4, "ctx": 8320, "block": 0},
        # The head of a four-sequence decode step: final norm, logits, greedy token.
        {"name": "head_int4_b4", "kind": "head", "shape": "8b", "fmt": "int4", "rows": 4},
        # A short chat turn: a few dozen tokens appended to a conversation.
        {"name": "prefill_int4_37", "kind": "prefill", "shape": "8b", "fmt": "int4", "m": 37, "start": 600},
        # The benchmark's prompt.
        {"name": "prefill_int4_512", "kind": "prefill", "shape": "8b", "fmt": "int4", "m": 512, "start": 0},
        # A medium prompt of a length that fills no tile, INT8 weights.
        {"name": "prefill_int8_300", "kind": "prefill", "shape": "8b", "fmt": "int8", "m": 300, "start": 0},
        # A long prompt, unquantized weights.
        {"name": "prefill_bf16_1000", "kind": "prefill", "shape": "8b", "fmt": "bf16", "m": 1000, "start": 0},
        # The last chunk of an 8192-token prompt prefilled in 2048-token chunks.
        {"name": "prefill_int4_2048_at_6144", "kind": "prefill", "shape": "8b", "fmt": "int4", "m": 2048, "start": 6144},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    fmt = rng.choice(["int4", "int4", "int8", "bf16"])
    shape = rng.choice(["8b", "8b", "8b", "2k"])
    block = rng.choice([0, 64])
    what = rng.random()
    if what < 0.34:
        return {"kind": "decode", "shape": shape, "fmt": fmt, "rows": _log_int(rng, 1, 16), "ctx": _log_int(rng, 64, 4096),
                "block": block}
    if what < 0.72:
        m = _log_int(rng, 9, 2048 if fmt == "int4" else 1500)
        return {"kind": "prefill", "shape": shape, "fmt": fmt, "m": m, "start": rng.choice([0, rng.randrange(0, 6145)])}
    if what < 0.81:
        return {"kind": "attention", "rows": _log_int(rng, 1, 8), "ctx": _log_int(rng, 512, 8320), "block": block}
    if what < 0.90:
        return {"kind": "head", "shape": shape, "fmt": fmt, "rows": _log_int(rng, 1, 16)}
    if what < 0.95:
        return {"kind": "session", "fmt": fmt, "layers": 2, "prompt": _log_int(rng, 16, 1024)}
    return {"kind": "generate", "prompt": _log_int(rng, 8, 200), "new": rng.randrange(8, 49)}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std, mean=0.0):
    """bf16 N(mean, std) values"""
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std + mean).to(torch.bfloat16)


def _dims(case):
    return SHAPES[case.get("shape", "8b")]


def _layer_weights(g, s):
    H, Q, KV, F = s["hidden"], s["hq"] * s["d"], s["hkv"] * s["d"], s["ffn"]
    w = {"qkv": (Q + 2 * KV, H), "o": (H, Q), "gate_up": (2 * F, H), "down": (H, F)}
    return {n: _normal(g, shape, 0.02) for n, shape in w.items()}


def _rope_tables(n, d):
    inv = THETA ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    a = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * inv[None, :]
    return a.cos().float(), a.sin().float()


def _positions(case):
    """The position each sequence decodes at: from ctx - 1 down to about half of it."""
    r, ctx = case["rows"], case["ctx"]
    return [ctx - 1 - i * (ctx // (2 * r)) for i in range(r)]


def _capacity(case):
    last = case["start"] + case["m"] if case["kind"] == "prefill" else case["ctx"]
    return -(-last // 256) * 256


def _cache(g, case, s):
    """K and V values [rows][hkv][capacity][d]; positions not reached yet hold zeros."""
    cap, d = _capacity(case), s["d"]
    if case["kind"] == "prefill":
        rows, filled = 1, [case["start"]]
    else:
        pos = _positions(case)
        rows, filled = len(pos), [p + (case["kind"] == "attention") for p in pos]
    kv = []
    for _ in range(2):
        t = torch.randn((rows, s["hkv"], cap, d), generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)
        for r, n in enumerate(filled):
            t[r, :, n:] = 0
        kv.append(t)
    return kv


def _inputs(case, seed):
    """Everything a case computes from, made with torch from the seed alone."""
    g, s, kind = _gen(seed), _dims(case), case["kind"]
    x = {}
    if kind in ("decode", "prefill"):
        rows = case["rows"] if kind == "decode" else case["m"]
        x["w"] = _layer_weights(g, s)
        x["embed"] = _normal(g, (EMBED_ROWS, s["hidden"]), 1.0)
        x["ids"] = torch.randint(0, EMBED_ROWS, (rows,), generator=g, device="cuda")
        x["norm1"], x["norm2"] = (_normal(g, (s["hidden"],), 0.25, 1.0) for _ in range(2))
        x["k"], x["v"] = _cache(g, case, s)
        x["cos"], x["sin"] = _rope_tables(_capacity(case), s["d"])
    elif kind == "attention":
        x["q"] = _normal(g, (case["rows"], s["hq"] * s["d"]), 1.0)
        x["k"], x["v"] = _cache(g, case, s)
    elif kind == "head":
        x["h"] = _normal(g, (case["rows"], s["hidden"]), 1.0)
        x["norm"] = _normal(g, (s["hidden"],), 0.25, 1.0)
        x["w"] = {"head": _normal(g, (s["vocab"], s["hidden"]), 0.02)}
    elif kind == "generate":
        t = TINY
        H, Q, KV, F, V = t["hidden"], t["hq"] * t["d"], t["hkv"] * t["d"], t["ffn"], t["vocab"]
        shapes = {"model.embed_tokens.weight": (V, H), "model.norm.weight": (H,), "lm_head.weight": (V, H)}
        for i in range(t["layers"]):
            p = "model.layers.%d." % i
            shapes.update({p + "input_layernorm.weight": (H,), p + "post_attention_layernorm.weight": (H,),
                           p + "self_attn.q_proj.weight": (Q, H), p + "self_attn.k_proj.weight": (KV, H),
                           p + "self_attn.v_proj.weight": (KV, H), p + "self_attn.o_proj.weight": (H, Q),
                           p + "mlp.gate_proj.weight": (F, H), p + "mlp.up_proj.weight": (F, H),
                           p + "mlp.down_proj.weight": (H, F)})
        x["w"] = {n: torch.randn(sh, generator=g, device="cuda") * (0.1 if len(sh) == 1 else 0.02) + (len(sh) == 1)
                  for n, sh in shapes.items()}
        x["prompt"] = torch.randint(0, V, (case["prompt"],), generator=g, device="cuda")
    else:
        x["prompt"] = torch.randint(0, s["vocab"], (case["prompt"],), generator=g, device="cuda")
    return x


# ------------------------------------------------------------------ what a program keeps
def _ptr(t):
    return t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _empty(*shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _scratch(nbytes):
    return torch.zeros(max(int(nbytes), 16), dtype=torch.uint8, device="cuda")


def _pack(src, fmt, keep):
    """The library's device weight of a bf16 matrix (the loader's conversion)."""
    L, (n, k) = N.lib(), src.shape
    db, sb = N.i64(), N.i64()
    L.call("am_gfx950_weight_bytes", n, k, fmt, GROUP, db, sb)
    data = torch.empty(db.value, dtype=torch.uint8, device="cuda")
    scales = torch.empty(max(sb.value, 16), dtype=torch.uint8, device="cuda")
    w = N.Weight(_ptr(data), _ptr(scales) if sb.value else None, n, k, fmt, GROUP)
    args = N.QuantizeArgs(_ptr(src), N.AM_DT_BF16, n, w, 0, 1)
    L.call("am_gfx950_pack_plain" if fmt == N.AM_WF_BF16 else "am_gfx950_quantize", args, _stream())
    keep += [data, scales]
    return w


def _paged(t, block):
    """Pools [blocks][hkv][block][d] and the block table of a contiguous cache, with the
    sequences' blocks interleaved as growing sequences take them."""
    rows, hkv, cap, d = t.shape
    per = cap // block
    pool = t.view(rows, hkv, per, block, d).permute(2, 0, 1, 3, 4).reshape(per * rows, hkv, block, d).contiguous()
    table = (torch.arange(per, device="cuda")[None, :] * rows + torch.arange(rows, device="cuda")[:, None]).to(torch.int32)
    return pool, table.contiguous()


class _Calls:
    """A frozen list of library calls with the buffers they use."""

    def __init__(self):
        self.keep, self.calls, self.out = [], [], {}

    def add(self, name, args):
        self.calls.append((name, args))

    def run(self):
        L, s = N.lib(), _stream()
        for name, args in self.calls:
            L.call(name, args, s)
        return self.out


def _plan_decode(case, x):
    p, s, L = _Calls(), _dims(case), N.lib()
    H, hq, hkv, d, F, rows, cap = s["hidden"], s["hq"], s["hkv"], s["d"], s["ffn"], case["rows"], _capacity(case)
    bf, w = N.AM_DT_BF16, {n: _pack(t, FORMATS[case["fmt"]], p.keep) for n, t in x["w"].items()}
    k, v, pages = x["k"], x["v"], None
    if case["block"]:
        (k, table), (v, _) = _paged(k, case["block"]), _paged(v, case["block"])
        pages = C.pointer(N.KvPages(_ptr(table), case["block"], table.shape[1], k.shape[0], None))
        p.keep.append(table)
    pos = torch.tensor(_positions(case), dtype=torch.int64, device="cuda")
    h, q, attn, act = _empty(rows, H), _empty(rows, hq * d), _empty(rows, hq * d), _empty(rows, F)
    wb = L.am_gfx950_attention_workspace_bytes(rows, 1, hq, hkv, d, cap, 0)
    ws, cbs = _scratch(wb), hkv * cap * d
    p.keep += [x["embed"], x["ids"], x["norm1"], x["norm2"], x["cos"], x["sin"], pos, ws]
    p.add("am_gfx950_embedding", N.EmbeddingArgs(_ptr(x["ids"]), N.AM_DT_I64, rows, _ptr(x["embed"]), bf, EMBED_ROWS, H,
                                                 _ptr(h), bf, None, 0))
    p.add("am_gfx950_fused_qkv", N.FusedQkvArgs(_ptr(h), _ptr(x["norm1"]), EPS, w["qkv"], _ptr(x["cos"]), _ptr(x["sin"]),
                                                _ptr(pos), _ptr(q), _ptr(k), _ptr(v), hq, hkv, d, cap, bf, rows, cbs, pages))
    p.add("am_gfx950_attention", N.AttentionArgs(_ptr(q), _ptr(k), _ptr(v), _ptr(attn), 1, hq, hkv, d, cap, 0, _ptr(pos),
                                                 rows, cbs, bf, 0, _ptr(ws), wb, pages))
    p.add("am_gfx950_fused_linear_residual", N.FusedLinearResidualArgs(_ptr(attn), w["o"], _ptr(h), bf, rows))
    p.add("am_gfx950_fused_gate_up", N.FusedGateUpArgs(_ptr(h), _ptr(x["norm2"]), EPS, w["gate_up"], _ptr(act), bf, rows))
    p.add("am_gfx950_fused_linear_residual", N.FusedLinearResidualArgs(_ptr(act), w["down"], _ptr(h), bf, rows))
    p.out = {"h": h, "q": q, "attn": attn, "act": act, "k": k, "v": v}
    return p


def _plan_prefill(case, x):
    p, s, L = _Calls(), _dims(case), N.lib()
    H, hq, hkv, d, F, m, cap = s["hidden"], s["hq"], s["hkv"], s["d"], s["ffn"], case["m"], _capacity(case)
    bf, w = N.AM_DT_BF16, {n: _pack(t, FORMATS[case["fmt"]], p.keep) for n, t in x["w"].items()}
    k, v = x["k"], x["v"]
    start = torch.tensor([case["start"]], dtype=torch.int64, device="cuda")
    h, xn, q, attn, act = _empty(m, H), _empty(m, H), _empty(m, hq * d), _empty(m, hq * d), _empty(m, F)
    gb = max(L.am_gfx950_gemm_workspace_bytes(m, wt.n, wt.k, GROUP) for wt in w.values())
    ab = L.am_gfx950_attention_workspace_bytes(1, m, hq, hkv, d, cap, 0)
    gws, aws = _scratch(gb), _scratch(ab)
    g = (_ptr(gws), gb) if gb else (None, 0)
    none3, none2 = lambda *o: (N.vp * 3)(*o), (N.i64 * 2)(0, 0)  # noqa: E731
    rope = N.PrefillRopeKv(_ptr(x["cos"]), _ptr(x["sin"]), cap, _ptr(start), _ptr(k), _ptr(v), hq, hkv, d, cap, None, None)
    p.keep += [x["embed"], x["ids"], x["norm1"], x["norm2"], x["cos"], x["sin"], start, xn, gws, aws, rope]
    p.add("am_gfx950_embedding", N.EmbeddingArgs(_ptr(x["ids"]), N.AM_DT_I64, m, _ptr(x["embed"]), bf, EMBED_ROWS, H,
                                                 _ptr(h), bf, None, 0))
    p.add("am_gfx950_rmsnorm", N.RmsNormArgs(_ptr(h), _ptr(x["norm1"]), _ptr(xn), m, H, H, H, EPS, bf, bf, bf))
    p.add("am_gfx950_prefill_linear", N.PrefillLinearArgs(_ptr(xn), m, w["qkv"], N.AM_PREFILL_QKV_ROPE_KV,
                                                          none3(_ptr(q), None, None), none2, g[0], g[1], C.pointer(rope)))
    p.add("am_gfx950_attention", N.AttentionArgs(_ptr(q), _ptr(k), _ptr(v), _ptr(attn), m, hq, hkv, d, cap, 0, _ptr(start),
                                                 1, 0, bf, 0, _ptr(aws) if ab else None, ab, None))
    p.add("am_gfx950_linear", N.LinearArgs(_ptr(attn), bf, m, w["o"], _ptr(h), bf, _ptr(h), 2, g[0], g[1]))
    p.add("am_gfx950_rmsnorm", N.RmsNormArgs(_ptr(h), _ptr(x["norm2"]), _ptr(xn), m, H, H, H, EPS, bf, bf, bf))
    p.add("am_gfx950_prefill_linear", N.PrefillLinearArgs(_ptr(xn), m, w["gate_up"], N.AM_PREFILL_SILU_MUL,
                                                          none3(_ptr(act), None, None), none2, g[0], g[1], None))
    p.add("am_gfx950_linear", N.LinearArgs(_ptr(act), bf, m, w["down"], _ptr(h), bf, _ptr(h), 2, g[0], g[1]))
    p.out = {"h": h, "q": q, "attn": attn, "act": act, "k": k, "v": v}
    return p


def _plan_attention(case, x):
    p, s, L = _Calls(), _dims(case), N.lib()
    hq, hkv, d, rows, cap = s["hq"], s["hkv"], s["d"], case["rows"], _capacity(case)
    k, v, pages = x["k"], x["v"], None
    if case["block"]:
        (k, table), (v, _) = _paged(k, case["block"]), _paged(v, case["block"])
        pages = C.pointer(N.KvPages(_ptr(table), case["block"], table.shape[1], k.shape[0], None))
        p.keep.append(table)
    pos = torch.tensor(_positions(case), dtype=torch.int64, device="cuda")
    attn, wb = _empty(rows, hq * d), L.am_gfx950_attention_workspace_bytes(rows, 1, hq, hkv, d, cap, 0)
    ws = _scratch(wb)
    p.keep += [x["q"], k, v, pos, ws]
    p.add("am_gfx950_attention", N.AttentionArgs(_ptr(x["q"]), _ptr(k), _ptr(v), _ptr(attn), 1, hq, hkv, d, cap, 0, _ptr(pos),
                                                 rows, hkv * cap * d, N.AM_DT_BF16, 0, _ptr(ws), wb, pages))
    p.out = {"attn": attn}
    return p


def _plan_head(case, x):
    p, s, L, rows = _Calls(), _dims(case), N.lib(), case["rows"]
    w = _pack(x["w"]["head"], FORMATS[case["fmt"]], p.keep)
    wb = L.am_gfx950_lm_head_workspace_bytes()
    logits, token, ws = _empty(rows, s["vocab"], dtype=torch.float32), _empty(rows, dtype=torch.int64), _scratch(wb)
    p.keep += [x["h"], x["norm"], ws]
    p.add("am_gfx950_fused_lm_head", N.FusedLmHeadArgs(_ptr(x["h"]), _ptr(x["norm"]), EPS, w, _ptr(logits), _ptr(token), None,
                                                       None, None, N.AM_DT_BF16, _ptr(ws), wb, rows, 0))
    p.out = {"logits": logits, "token": token}
    return p


class _Session:
    """A runtime, a model and one single-sequence session, released with the object."""

    def __init__(self, open_model, vocab, prompt, new):
        L = N.lib()
        self.rt, self.model, self.session = N.vp(), N.vp(), N.vp()
        L.call("am_runtime_open", 0, C.byref(self.rt))
        open_model(self.rt, C.byref(self.model))
        L.call("am_session_open", self.model, C.byref(N.SessionOptions(1, 1)), C.byref(self.session))
        self.prompt = prompt.cpu().numpy().astype(np.int64)
        self.new, self.tokens, self.logits = new, np.zeros(max(new, 1), np.int64), np.zeros(vocab, np.float32)

    def run(self):
        L, n = N.lib(), N.i64()
        if self.new:  # prompt in, greedy tokens out
            L.call("am_session_generate_ids", self.session, self.prompt.ctypes.data, self.prompt.size, self.new, -1,
                   self.tokens.ctypes.data, C.byref(n))
        else:  # first token of a prompt
            L.call("am_session_prefill", self.session, self.prompt.ctypes.data, self.prompt.size, C.byref(n))
            self.tokens[0] = n.value
        L.call("am_session_logits", self.session, self.logits.ctypes.data)
        return {"tokens": self.tokens, "logits": self.logits}

    def __del__(self):
        L = N.lib()
        for name, handle in (("am_session_destroy", self.session), ("am_model_destroy", self.model),
                             ("am_runtime_destroy", self.rt)):
            if handle:
                getattr(L, name)(handle)


def _write_checkpoint(folder, weights):
    t = TINY
    config = {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "hidden_size": t["hidden"],
              "intermediate_size": t["ffn"], "num_hidden_layers": t["layers"], "num_attention_heads": t["hq"],
              "num_key_value_heads": t["hkv"], "head_dim": t["d"], "vocab_size": t["vocab"], "rms_norm_eps": EPS,
              "rope_theta": t["theta"], "max_position_embeddings": 2048, "tie_word_embeddings": False,
              "torch_dtype": "float32", "hidden_act": "silu"}
    with open(os.path.join(folder, "config.json"), "w") as f:
        json.dump(config, f)
    header, at = {}, 0
    for name, w in weights.items():
        header[name] = {"dtype": "F32", "shape": list(w.shape), "data_offsets": [at, at + w.numel() * 4]}
        at += w.numel() * 4
    text = json.dumps(header).encode()
    with open(os.path.join(folder, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for w in weights.values():
            f.write(memoryview(w.cpu().numpy()).cast("B"))


def _session(case, x, seed):
    if case["kind"] == "generate":
        def load(rt, out):
            with tempfile.TemporaryDirectory() as folder:
                _write_checkpoint(folder, x["w"])
                opt = N.ModelLoadOptions(N.AM_DT_F32, N.AM_WF_F32, GROUP, 256, 128)
                N.lib().call("am_model_load_hf", rt, folder.encode(), C.byref(opt), out)
        return _Session(load, TINY["vocab"], x["prompt"], case["new"])
    s = SHAPES["8b"]

    def create(rt, out):
        cfg = N.ModelConfig(case["layers"], s["hidden"], s["hq"], s["hkv"], s["d"], s["ffn"], s["vocab"], EPS, THETA,
                            N.AM_DT_BF16, FORMATS[case["fmt"]], GROUP, 2048, 512)
        N.lib().call("am_model_create_synthetic", rt, C.byref(cfg), seed, out)
    return _Session(create, s["vocab"], x["prompt"], 0)


def prepare(case, seed):
    x = _inputs(case, seed)
    plan = {"decode": _plan_decode, "prefill": _plan_prefill, "attention": _plan_attention, "head": _plan_head}.get(case["kind"])
    if plan is None:
        return _session(case, x, seed)
    p = plan(case, x)
    torch.cuda.synchronize()  # the unpacked weights may go once they are packed
    return p


def run(state):
    return state.run()


# ------------------------------------------------------------------ the work and its bounds
def _weight_bytes(n, k, fmt):
    return {"int4": n * k / 2 + n * k / GROUP * 2, "int8": n * k + 4 * n, "bf16": 2 * n * k}[fmt]


def _layer_work(s, fmt, rows, contexts, kv_rows, kv_read):
    """One layer: weights and cache read once, activations and new cache rows once."""
    H, Q, KV, F = s["hidden"], s["hq"] * s["d"], s["hkv"] * s["d"], s["ffn"]
    shapes = [(Q + 2 * KV, H), (H, Q), (2 * F, H), (H, F)]
    b = sum(_weight_bytes(n, k, fmt) for n, k in shapes) + rows * H * 2 * 2 + kv_rows * KV * 4 + kv_read * KV * 4
    return {"bytes": b, "flops": 2 * rows * sum(n * k for n, k in shapes) + 4 * Q * contexts}


def work(case):
    s, kind = _dims(case), case["kind"]
    if kind == "decode":
        ctx = sum(p + 1 for p in _positions(case))
        return _layer_work(s, case["fmt"], case["rows"], ctx, case["rows"], ctx)
    if kind == "prefill":
        m, a = case["m"], case["start"]
        return _layer_work(s, case["fmt"], m, m * a + m * (m + 1) // 2, m, a)
    if kind == "attention":
        ctx, Q = sum(p + 1 for p in _positions(case)), s["hq"] * s["d"]
        return {"bytes": ctx * s["hkv"] * s["d"] * 4 + case["rows"] * Q * 4, "flops": 4 * Q * ctx}
    if kind == "head":
        n, k = s["vocab"], s["hidden"]
        return {"bytes": _weight_bytes(n, k, case["fmt"]) + case["rows"] * (2 * k + 4 * n), "flops": 2 * case["rows"] * n * k}
    if kind == "session":
        m = case["prompt"]
        w = _layer_work(s, case["fmt"], m, m * (m + 1) // 2, m, 0)
        n, k = s["vocab"], s["hidden"]
        return {"bytes": case["layers"] * w["bytes"] + _weight_bytes(n, k, case["fmt"]) + 4 * n,
                "flops": case["layers"] * w["flops"] + 2 * n * k}
    t, m, new = TINY, case["prompt"], case["new"]
    layer = t["hidden"] * (2 * t["hq"] + 2 * t["hkv"]) * t["d"] + 3 * t["hidden"] * t["ffn"]
    head = t["vocab"] * t["hidden"]
    return {"bytes": 4.0 * new * (t["layers"] * layer + head),
            "flops": 2.0 * ((m + new - 1) * t["layers"] * layer + new * head)}


def tolerance(case):
    if case["kind"] == "generate":  # fp32 sums; a greedy token flips only on an fp32 tie
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.01}
    if case["kind"] == "head":  # fp32 logits of bf16 products
        return {"rel": 1e-2, "max": 0.1, "differ": 0.01}
    if case["kind"] == "session":  # rounding differences travel through both layers
        return {"rel": 2e-2, "max": 0.2, "differ": 0.01}
    return {"rel": 1e-2, "max": 0.2}


# ------------------------------------------------------------------ 64-bit results
def _dequant(w, fmt):
    """The weight values a format holds for a bf16 matrix, in 64 bits."""
    w = w.float()
    if fmt == "int8":
        s = w.abs().amax(1, keepdim=True) / 127.0
        s = torch.where(s == 0, torch.ones_like(s), s)
        return (w / s).round().clamp(-127, 127).double() * s.double()
    if fmt == "int4":
        n, k = w.shape
        g = w.view(n, k // GROUP, GROUP)
        s = (g.abs().amax(2, keepdim=True) / 7.0).half().float()
        q = torch.where(s == 0, torch.zeros_like(g), (g / s).round().clamp(-8, 7))
        return (q.double() * s.double()).view(n, k)
    return w.double()


def _norm(x, w, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rotate(x, cos, sin):
    """x [rows][heads][d] at the positions whose table rows are given"""
    h = x.shape[-1] // 2
    a, b, c, s = x[..., :h], x[..., h:], cos.double()[:, None], sin.double()[:, None]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, start):
    """q [m][hq][d] at positions start + i over k, v [hkv][positions][d]"""
    m, hq, d = q.shape
    g, n, out = hq // k.shape[0], k.shape[1], torch.empty_like(q)
    mask = torch.arange(n, device="cuda")[None, :] > start + torch.arange(m, device="cuda")[:, None]
    for h in range(hq):
        sc = (q[:, h] @ k[h // g].T.contiguous() / math.sqrt(d)).masked_fill(mask, -math.inf)
        out[:, h] = torch.softmax(sc, -1) @ v[h // g]
    return out


def _exact_layer(case, seed):
    x, s, fmt = _inputs(case, seed), _dims(case), case["fmt"]
    hq, hkv, d, F = s["hq"], s["hkv"], s["d"], s["ffn"]
    Q, KV = hq * d, hkv * d
    h = x["embed"].double()[x["ids"]]
    k, v = x["k"].double(), x["v"].double()
    rows = h.shape[0]
    qkv = _norm(h, x["norm1"]) @ _dequant(x["w"]["qkv"], fmt).T
    if case["kind"] == "decode":
        seqs = [(r, p, r, r + 1) for r, p in enumerate(_positions(case))]  # sequence, position, its rows
    else:
        seqs = [(0, case["start"], 0, rows)]
    q_out, attn = torch.empty(rows, Q, dtype=torch.float64, device="cuda"), torch.empty(rows, Q, dtype=torch.float64, device="cuda")
    for b, p, r0, r1 in seqs:
        m = r1 - r0
        cos, sin = x["cos"][p:p + m], x["sin"][p:p + m]
        q = _rotate(qkv[r0:r1, :Q].reshape(m, hq, d), cos, sin)
        k[b, :, p:p + m] = _rotate(qkv[r0:r1, Q:Q + KV].reshape(m, hkv, d), cos, sin).transpose(0, 1)
        v[b, :, p:p + m] = qkv[r0:r1, Q + KV:].reshape(m, hkv, d).transpose(0, 1)
        q_out[r0:r1] = q.reshape(m, Q)
        attn[r0:r1] = _attend(q, k[b, :, :p + m], v[b, :, :p + m], p).reshape(m, Q)
    h = h + attn @ _dequant(x["w"]["o"], fmt).T
    gu = _norm(h, x["norm2"]) @ _dequant(x["w"]["gate_up"], fmt).T
    act = torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]
    h = h + act @ _dequant(x["w"]["down"], fmt).T
    if case.get("block"):
        k, v = _paged(k, case["block"])[0], _paged(v, case["block"])[0]
    return {"h": h, "q": q_out, "attn": attn, "act": act, "k": k, "v": v}


def _exact_generate(case, seed):
    x, t = _inputs(case, seed), TINY
    w = {n: a.double() for n, a in x["w"].items()}
    hq, hkv, d = t["hq"], t["hkv"], t["d"]
    total = case["prompt"] + case["new"]
    inv = t["theta"] ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    ang = torch.arange(total, device="cuda", dtype=torch.float64)[:, None] * inv
    cos, sin = ang.cos(), ang.sin()
    caches = [[torch.zeros(hkv, total, d, dtype=torch.float64, device="cuda") for _ in range(2)] for _ in range(t["layers"])]
    ids, at, tokens, logits = x["prompt"], 0, [], None
    for _ in range(case["new"]):
        m = ids.numel()
        h = w["model.embed_tokens.weight"][ids]
        for i in range(t["layers"]):
            p, (k, v) = "model.layers.%d." % i, caches[i]
            a = _norm(h, w[p + "input_layernorm.weight"])
            q = _rotate((a @ w[p + "self_attn.q_proj.weight"].T).view(m, hq, d), cos[at:at + m], sin[at:at + m])
            k[:, at:at + m] = _rotate((a @ w[p + "self_attn.k_proj.weight"].T).view(m, hkv, d), cos[at:at + m],
                                      sin[at:at + m]).transpose(0, 1)
            v[:, at:at + m] = (a @ w[p + "self_attn.v_proj.weight"].T).view(m, hkv, d).transpose(0, 1)
            o = _attend(q, k[:, :at + m], v[:, :at + m], at).reshape(m, hq * d)
            h = h + o @ w[p + "self_attn.o_proj.weight"].T
            a = _norm(h, w[p + "post_attention_layernorm.weight"])
            act = torch.nn.functional.silu(a @ w[p + "mlp.gate_proj.weight"].T) * (a @ w[p + "mlp.up_proj.weight"].T)
            h = h + act @ w[p + "mlp.down_proj.weight"].T
        logits = _norm(h[-1], w["model.norm.weight"]) @ w["lm_head.weight"].T
        ids = logits.argmax().view(1)
        tokens.append(int(ids))
        at += m
    return {"tokens": None, "logits": logits}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_layer(case, seed)
    if kind == "attention":
        x, s = _inputs(case, seed), _dims(case)
        q = x["q"].double().view(case["rows"], s["hq"], s["d"])
        rows = [_attend(q[r:r + 1], x["k"][r, :, :p + 1].double(), x["v"][r, :, :p + 1].double(), p)
                for r, p in enumerate(_positions(case))]
        return {"attn": torch.cat(rows).reshape(case["rows"], -1)}
    if kind == "head":
        x = _inputs(case, seed)
        return {"logits": _norm(x["h"].double(), x["norm"]) @ _dequant(x["w"]["head"], case["fmt"]).T, "token": None}
    if kind == "generate":
        return _exact_generate(case, seed)
    return None  # the session's weights are made by the library's own generator
