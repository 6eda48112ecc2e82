"""Timed cases of the library's public entry points on one GPU: single operators, stacks of decoder layers, and the
two whole-model calls (greedy decode and a 2048-token prompt).

A case is a dict of plain values whose "kind" names the entry point:
  gemv, qmm             one projection at decode, fp16 or group-quantized (soc_gemv_f16, soc_qmm)
  sample                top-k candidates of one logits row (soc_sample_topk)
  attn_decode           one token's attention over a KV cache (soc_attention_decode)
  attn_prefill          a prompt chunk's causal attention (soc_attention_prefill)
  prompt                soc_forward over n tokens of a stack of layers behind `past` cached positions
  decode                one sequence, `steps` greedy steps on the device and one more that returns its logits
  batch                 one step of n sequences of different lengths (soc_decode_batch)
Layer widths are the dense Qwen3 sizes of soc_amd; stacks of a few layers with a 16384-word head stand for the model's
layers, since a change of rounding in one layer travels through all that follow.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import soc_amd as S
from soc_amd.capi import check, lib

SHAPES = {"0.6b": S.QWEN3_0_6B, "1.7b": S.QWEN3_1_7B, "4b": S.QWEN3_4B, "8b": S.QWEN3_8B}
HEAD_WORDS = 16384  # vocabulary of the layer stacks


def listed():
    return [
        # one decode projection of a small model: the shortest call, where the launch counts
        {"name": "gemv gate 1.7b", "kind": "gemv", "n": 6144, "k": 2048},
        # the same call group-quantized, eight rows (a verification or small-batch step)
        {"name": "int4 down 0.6b x 8", "kind": "qmm", "bits": 4, "m": 8, "n": 1024, "k": 3072},
        # the sampler behind every sampled token: candidates of one row of the full vocabulary
        {"name": "sample top 50", "kind": "sample", "vocab": 151936, "k": 50, "temperature": 0.7},
        # decode attention late in a long conversation, 32 query heads on 8 KV heads
        {"name": "attention decode 4071", "kind": "attn_decode", "len": 4071, "cap": 4160, "nq": 32, "nkv": 8},
        # attention of a long prompt
        {"name": "attention prefill 2048", "kind": "attn_prefill", "rows": 2048, "past": 0, "nq": 16, "nkv": 8},
        # a chat turn's prompt: a few dozen tokens, an odd number of them
        {"name": "prompt 31 0.6b", "kind": "prompt", "shape": "0.6b", "layers": 4, "bits": 0, "n": 31, "past": 0,
         "logit_rows": 1},
        # a follow-up turn of a larger model behind a cached conversation, ragged on every tile
        {"name": "prompt 333 after 700 4b", "kind": "prompt", "shape": "4b", "layers": 2, "bits": 0, "n": 333,
         "past": 700, "logit_rows": 1},
        # the whole small model on a long prompt
        {"name": "prefill 2048 0.6b whole", "kind": "prompt", "shape": "0.6b", "layers": 28, "bits": 0, "n": 2048,
         "past": 0, "logit_rows": 1},
        # the whole small model generating for one user
        {"name": "decode 0.6b whole", "kind": "decode", "shape": "0.6b", "layers": 28, "bits": 0, "past": 97,
         "steps": 31},
        # single-sequence generation with int4 projections
        {"name": "decode int4 0.6b", "kind": "decode", "shape": "0.6b", "layers": 4, "bits": 4, "past": 300,
         "steps": 15},
        # sixteen users of different lengths on a larger model
        {"name": "batch 16 4b", "kind": "batch", "shape": "4b", "layers": 4, "n": 16, "longest": 4096},
        # a busier server on the small model: more rows than one weight tile takes
        {"name": "batch 100 0.6b", "kind": "batch", "shape": "0.6b", "layers": 4, "n": 100, "longest": 1000},
    ]


def _spread(rng, lo, hi, step=1):
    """A size between lo and hi, even over its logarithm, a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["gemv", "qmm", "sample", "attn_decode", "attn_prefill", "prompt", "prompt", "decode", "decode",
                       "batch", "batch"])
    if kind == "gemv":
        n = _spread(rng, 1000, 152000)
        return {"kind": kind, "n": n, "k": _spread(rng, 512, 12288 if n < 32768 else 4096, 8)}
    if kind == "qmm":
        m = rng.choice([1, 2, 4, 8])
        return {"kind": kind, "bits": rng.choice([4, 8]), "m": m, "n": _spread(rng, 1000, 152000),
                "k": _spread(rng, 512, min(8192, 40960 // m), 64)}  # soc_qmm takes m * k up to 40960
    if kind == "sample":
        return {"kind": kind, "vocab": _spread(rng, 4096, 151936), "k": rng.choice([1, 2, 8, 20, 40, 50, 64]),
                "temperature": rng.choice([0.6, 0.7, 1.0])}
    heads = rng.choice([(16, 8), (32, 8), (16, 8), (8, 8)])
    if kind == "attn_decode":
        n = _spread(rng, 16, 9000)
        return {"kind": kind, "len": n, "cap": n + rng.randrange(1, 600), "nq": heads[0], "nkv": heads[1]}
    if kind == "attn_prefill":
        return {"kind": kind, "rows": _spread(rng, 2, 3000), "past": rng.choice([0, 0, rng.randrange(1, 1200)]),
                "nq": heads[0], "nkv": heads[1]}
    shape = rng.choice(sorted(SHAPES))
    if kind == "prompt":
        n = _spread(rng, 2, 2048)
        return {"kind": kind, "shape": shape, "layers": rng.choice([1, 2]), "bits": 0, "n": n,
                "past": rng.choice([0, 0, rng.randrange(1, 1500)]), "logit_rows": min(n, rng.choice([1, 1, 1, 5]))}
    if kind == "decode":
        bits = rng.choice([0, 0, 4, 8]) if shape in ("0.6b", "1.7b") else 0
        return {"kind": kind, "shape": shape, "layers": rng.choice([2, 3, 4]), "bits": bits,
                "past": _spread(rng, 16, 3000), "steps": rng.randrange(3, 24)}
    return {"kind": kind, "shape": shape, "layers": rng.choice([2, 3]), "n": _spread(rng, 2, 256),
            "longest": _spread(rng, 200, 2500)}


# ---- inputs ----------------------------------------------------------------------------------------------------
_ctx = None


def _context():
    """The program's one device context."""
    global _ctx
    if _ctx is None:
        _ctx = S.Context(0)
    return _ctx


class _Plane:
    """A KV slot's fp16 plane in the engine's device memory, for torch.as_tensor; it keeps the engine alive."""

    def __init__(self, engine, ptr, shape):
        self.engine = engine
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f2", "data": (ptr, False), "version": 2}


class _Engine:
    """A model with its KV cache, released with the state that holds it."""

    def __init__(self, cfg, slots, capacity):
        self.cfg = cfg
        self.model = S.Model(_context(), cfg)
        self.slots, self.capacity, self.kv = slots, capacity, None

    def __del__(self):
        if self.kv is not None:
            self.kv.close()
        self.model.close()

    def cached(self, slot, layer, length):
        """The first `length` cached keys and values [kv heads][length][128] of a slot and layer, as tensors over the
        cache itself that hold the engine: its memory lasts as long as they do."""
        k, v = C.c_void_p(), C.c_void_p()
        check(lib().soc_kv_layer_planes(self.kv.h, slot, layer, C.byref(k), C.byref(v)))
        shape = (self.cfg.num_key_value_heads, self.capacity, 128)
        views = [torch.as_tensor(_Plane(self, p.value, shape), device="cuda")[:, :length] for p in (k, v)]
        for t in views:
            t.engine = self
        return views


def _config(case):
    full = SHAPES[case["shape"]]
    whole = case["layers"] == full.num_hidden_layers
    return S.QwenConfig(vocab_size=full.vocab_size if whole else HEAD_WORDS, hidden_size=full.hidden_size,
                        num_hidden_layers=case["layers"], num_attention_heads=full.num_attention_heads,
                        num_key_value_heads=full.num_key_value_heads, intermediate_size=full.intermediate_size,
                        max_position_embeddings=4608, tie_word_embeddings=True)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, sigma=1.0, dtype=torch.float16):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * sigma).to(dtype)


def _weights(cfg, seed):
    """Initialised as such models are: N(0, 0.02), the projections into the residual stream scaled by the depth, gains
    around one. The embedding (and tied head) is N(0, 0.05), so that, as in a trained model, the best next token
    stands well clear of the others and a generated sequence does not hang on the last bits of a logit."""
    g = _generator(seed)
    for name, shape in S.tensor_specs(cfg):
        if name.endswith("norm.weight"):
            w = (1.0 + 0.1 * torch.randn(shape, generator=g, device="cuda")).to(torch.float16)
        elif name.endswith(("o_proj.weight", "down_proj.weight")):
            w = _normal(g, shape, 0.02 / math.sqrt(2 * cfg.num_hidden_layers))
        else:
            w = _normal(g, shape, 0.05 if "embed" in name else 0.02)
        yield name, w


def _past(cfg, seed, slot, layer, length):
    """Cached keys and values [length][kv heads][128] of one slot and layer: keys of the normed scale, N(0, 1)."""
    g = _generator(seed * 1000003 + slot * 61 + layer + 1)
    return [_normal(g, (length, cfg.num_key_value_heads, 128)) for _ in range(2)]


def _tokens(case, seed, vocab, n):
    return np.random.RandomState(seed).randint(0, vocab, n).astype(np.int32)


def _lengths(case, seed):
    """Lengths of the batch's sequences, from a 64th of the longest up."""
    r = np.random.RandomState(seed + 7)
    return r.randint(max(1, case["longest"] // 64), case["longest"] + 1, case["n"]).tolist()


def _engine(case, seed, slots, capacity, lengths):
    cfg = _config(case)
    e = _Engine(cfg, slots, capacity)
    for name, w in _weights(cfg, seed):
        torch.cuda.synchronize()
        check(lib().soc_model_load_tensor_device(e.model.h, name.encode(), w.data_ptr(), 1, w.numel()))
    check(lib().soc_model_finalize(e.model.h))
    if case.get("bits"):
        e.model.quantize(case["bits"])
    e.kv = S.KVCache(e.model, slots, capacity)
    for slot, length in enumerate(lengths):
        for layer in range(cfg.num_hidden_layers if length else 0):
            k, v = _past(cfg, seed, slot, layer, length)
            torch.cuda.synchronize()
            check(lib().soc_kv_append(e.kv.h, slot, layer, 0, length, k.data_ptr(), v.data_ptr(), 1))
        check(lib().soc_kv_set_length(e.kv.h, slot, length))
    return e


def _floats(*shape):
    return torch.zeros(shape, device="cuda", dtype=torch.float32)


def _op_inputs(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind == "gemv":
        return {"w": _normal(g, (case["n"], case["k"]), 0.02), "x": _normal(g, (case["k"],))}
    if kind == "qmm":
        n, k, q = case["n"], case["k"], 127 if case["bits"] == 8 else 7
        codes = torch.randint(-q, q + 1, (n, k), generator=g, device="cuda", dtype=torch.int8)
        scales = (0.06 / q * (0.5 + torch.rand((n, k // 64), generator=g, device="cuda"))).to(torch.float16)
        return {"codes": codes, "scales": scales, "x": _normal(g, (case["m"], k))}
    if kind == "sample":
        return {"row": _normal(g, (case["vocab"],), 2.0, torch.float32)}
    rows, cap = (1, case["cap"]) if kind == "attn_decode" else (case["rows"], case["past"] + case["rows"])
    return {"q": _normal(g, (rows, case["nq"], 128), 1.0, torch.float32), "k": _normal(g, (case["nkv"], cap, 128)),
            "v": _normal(g, (case["nkv"], cap, 128))}


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "ctx": _context()}
    if kind in ("gemv", "qmm", "sample", "attn_decode", "attn_prefill"):
        s.update(_op_inputs(case, seed))
        if kind == "qmm":
            if case["bits"] == 4:  # two codes a byte, the even k in the low nibble
                c = s["codes"]
                s["codes"] = (c[:, 0::2] & 15) | (c[:, 1::2] << 4)
            s["y"] = _floats(case["m"], case["n"])
        elif kind == "gemv":
            s["y"] = _floats(case["n"])
        elif kind != "sample":
            s["out"] = torch.zeros_like(s["q"])
    elif kind == "batch":
        lengths = _lengths(case, seed)
        s["engine"] = e = _engine(case, seed, case["n"], case["longest"] + 64, lengths)
        s["lengths"], s["slots"] = lengths, np.arange(case["n"], dtype=np.int32)
        s["ids"] = _tokens(case, seed, e.cfg.vocab_size, case["n"])
        s["logits"] = _floats(case["n"], e.cfg.vocab_size)
        s["next"] = np.zeros(case["n"], np.int32)
    else:
        new = case["n"] if kind == "prompt" else case["steps"] + 1
        s["engine"] = e = _engine(case, seed, 1, case["past"] + new + 32, [case["past"]])
        s["ids"] = _tokens(case, seed, e.cfg.vocab_size, new)
        s["logits"] = _floats(case.get("logit_rows", 1), e.cfg.vocab_size)
        if kind == "prompt":
            s["hidden"] = _floats(case["n"], e.cfg.hidden_size)
        else:
            s["tokens"] = np.zeros(case["steps"], np.int32)
        # the last layer's cache: it depends on what every layer before it did
        s["keys"], s["values"] = e.cached(0, case["layers"] - 1, case["past"] + new)
    torch.cuda.synchronize()
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------
def run(s):
    case, L = s["case"], lib()
    kind = case["kind"]
    if kind == "gemv":
        S.gemv_f16(s["ctx"], s["w"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(), case["n"], case["k"])
        return s["y"]
    if kind == "qmm":
        S.qmm(s["ctx"], s["x"].data_ptr(), s["codes"].data_ptr(), case["bits"], s["scales"].data_ptr(),
              s["y"].data_ptr(), case["m"], case["n"], case["k"])
        return s["y"]
    if kind == "sample":
        token, ids, values = S.sample_topk(s["ctx"], s["row"].data_ptr(), case["vocab"], case["k"],
                                           case["temperature"])
        return {"token": token, "ids": ids, "values": values}
    if kind == "attn_decode":
        S.attention_decode(s["ctx"], s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["out"].data_ptr(),
                           case["len"], case["nq"], case["nkv"], case["cap"])
        return s["out"]
    if kind == "attn_prefill":
        S.attention_prefill(s["ctx"], s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), s["out"].data_ptr(),
                            case["rows"], case["past"], case["nq"], case["nkv"], case["past"] + case["rows"])
        return s["out"]
    e = s["engine"]
    m, kv = e.model.h, e.kv.h
    if kind == "batch":
        for slot, length in enumerate(s["lengths"]):  # the same step again: the sequences back at their lengths
            check(L.soc_kv_set_length(kv, slot, length))
        check(L.soc_decode_batch(m, kv, case["n"], s["slots"].ctypes.data, s["ids"].ctypes.data,
                                   s["logits"].data_ptr(), s["next"].ctypes.data))
        return {"logits": s["logits"], "next": s["next"]}
    check(L.soc_kv_set_length(kv, 0, case["past"]))
    token = C.c_int32()
    if kind == "prompt":
        check(L.soc_forward(m, kv, 0, s["ids"].ctypes.data, case["n"], case["past"], s["hidden"].data_ptr(),
                              case["logit_rows"], s["logits"].data_ptr(), C.byref(token)))
        return {"hidden": s["hidden"], "logits": s["logits"], "token": token.value, "keys": s["keys"],
                "values": s["values"]}
    check(L.soc_decode_steps(m, kv, 0, int(s["ids"][0]), case["steps"], s["tokens"].ctypes.data))
    check(L.soc_decode(m, kv, 0, int(s["tokens"][-1]), s["logits"].data_ptr(), C.byref(token)))
    return {"tokens": s["tokens"], "token": token.value, "logits": s["logits"], "keys": s["keys"],
            "values": s["values"]}


# ---- what a pass cannot do without --------------------------------------------------------------------------------
def _layer_weights(cfg):
    return (cfg.hidden_size * (2 * cfg.q_dim + 2 * cfg.kv_dim) + 3 * cfg.hidden_size * cfg.intermediate_size)


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        return {"bytes": 2 * case["n"] * case["k"] + 2 * case["k"] + 4 * case["n"], "flops": 2 * case["n"] * case["k"]}
    if kind == "qmm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": n * k * case["bits"] / 8 + n * k / 32 + 2 * m * k + 4 * m * n, "flops": 2 * m * n * k}
    if kind == "sample":
        return {"bytes": 4 * case["vocab"] + 8 * case["k"], "flops": case["vocab"]}
    if kind == "attn_decode":
        return {"bytes": 4 * case["len"] * case["nkv"] * 128 + 8 * case["nq"] * 128,
                "flops": 4 * case["nq"] * 128 * case["len"]}
    if kind == "attn_prefill":
        rows, past = case["rows"], case["past"]
        return {"bytes": 8 * rows * case["nq"] * 128 + 4 * (past + rows) * case["nkv"] * 128,
                "flops": 4 * case["nq"] * 128 * (rows * past + rows * (rows + 1) // 2)}
    cfg = _config(case)
    per_key = 4 * cfg.kv_dim * cfg.num_hidden_layers  # bytes of a cached position
    head = cfg.vocab_size * cfg.hidden_size
    weights = _layer_weights(cfg) * cfg.num_hidden_layers
    wbytes = weights * ({0: 2.0, 8: 1.0, 4: 0.5}[case.get("bits", 0)] + (1 / 32 if case.get("bits") else 0))
    attn = 4 * cfg.q_dim * cfg.num_hidden_layers  # flops per query and key
    if kind == "batch":
        keys = case["n"] * (case["longest"] + case["longest"] // 64) / 2
        return {"bytes": wbytes + 2 * head + per_key * (keys + case["n"]) + case["n"] * (2 * cfg.hidden_size +
                                                                                         4 * cfg.vocab_size),
                "flops": 2 * (weights + head) * case["n"] + attn * keys}
    past = case["past"]
    if kind == "decode":
        n = case["steps"] + 1
        keys = n * past + n * (n + 1) / 2
        return {"bytes": n * (wbytes + 2 * head + 2 * cfg.hidden_size) + per_key * (keys + n) + 4 * cfg.vocab_size,
                "flops": 2 * (weights + head) * n + attn * keys}
    n = case["n"]
    return {"bytes": wbytes + 2 * head + per_key * (past + 2 * n) + 6 * n * cfg.hidden_size +
            4 * case["logit_rows"] * cfg.vocab_size,
            "flops": 2 * weights * n + 2 * head * case["logit_rows"] + attn * (n * past + n * (n + 1) / 2)}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"  # candidates are picked, not computed
    # about four times the errors measured against exact() over the listed and drawn cases
    if kind in ("gemv", "qmm"):
        return {"rel": 1e-6}  # fp32 sums of exact products (1e-7)
    if kind in ("attn_decode", "attn_prefill"):
        return {"rel": 2e-6}  # fp32 softmax and sums over 16-bit keys and values (3e-7)
    if kind == "batch":
        return {"rel": 2e-4, "differ": 0.01}  # 32-bit activations, 16-bit keys and values (5e-5)
    # a prompt's projections read 16-bit activations (6e-4); a quantized model's too, at every step (7e-4)
    return {"rel": 3e-3, "differ": 0.01}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------
def _attend(q, k, v, past):
    """q [rows][nq][128], k / v [nkv][keys][128] in float64; row t sees keys 0 .. past + t."""
    rows, nq, nkv = q.shape[0], q.shape[1], k.shape[0]
    out = torch.empty_like(q)
    seen = torch.arange(k.shape[1], device=q.device)[None, :] <= past + torch.arange(rows, device=q.device)[:, None]
    for h in range(nq):
        kh, vh = k[h // (nq // nkv)], v[h // (nq // nkv)]
        sc = (q[:, h].contiguous() @ kh.t().contiguous()) / math.sqrt(128.0)
        out[:, h] = torch.softmax(sc.masked_fill(~seen, -math.inf), dim=-1) @ vh.contiguous()
    return out


def _norm(x, gain, eps=1e-6):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * gain


def _rope(x, pos, theta):
    i = torch.arange(64, device=x.device, dtype=torch.float64)
    a = pos.to(torch.float64)[:, None, None] / theta ** (2 * i / 128)
    c, s = torch.cos(a).float().double(), torch.sin(a).float().double()  # the table is 32-bit
    lo, hi = x[..., :64], x[..., 64:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _quantized(w, bits):
    """Group-64 codes times their fp16 scales (the packer's rule)."""
    q = 127 if bits == 8 else 7
    g = w.double().reshape(w.shape[0], -1, 64)
    sc = (g.abs().amax(-1, keepdim=True).float() / q).to(torch.float16).double()
    r = torch.where(sc > 0, g.float() * (1.0 / sc.float()), 0.0).double()  # the packer's 32-bit quotient
    codes = (torch.sign(r) * torch.floor(r.abs() + 0.5)).clamp(-q, q)
    return (codes * sc).reshape(w.shape)


def _forward(cfg, w, x, past_kv, pos0):
    """All layers over rows x [n][H] behind cached keys / values: rows out, and each layer's keys and values."""
    n, kv = x.shape[0], []
    pos = torch.arange(pos0, pos0 + n, device=x.device)
    for l in range(cfg.num_hidden_layers):
        p = f"model.layers.{l}."
        lin = lambda v, name: v @ w[p + name].double().t()  # noqa: E731
        h = _norm(x, w[p + "input_layernorm.weight"].double())
        q = lin(h, "self_attn.q_proj.weight").view(n, -1, 128)
        k = lin(h, "self_attn.k_proj.weight").view(n, -1, 128)
        v = lin(h, "self_attn.v_proj.weight").view(n, -1, 128)
        q = _rope(_norm(q, w[p + "self_attn.q_norm.weight"].double()), pos, cfg.rope_theta)
        k = _rope(_norm(k, w[p + "self_attn.k_norm.weight"].double()), pos, cfg.rope_theta)
        pk, pv = past_kv[l]
        k = torch.cat([pk, k.transpose(0, 1)], 1)
        v = torch.cat([pv, v.transpose(0, 1)], 1)
        kv.append((k, v))
        x = x + lin(_attend(q, k, v, k.shape[1] - n).reshape(n, -1), "self_attn.o_proj.weight")
        h = _norm(x, w[p + "post_attention_layernorm.weight"].double())
        x = x + lin(torch.nn.functional.silu(lin(h, "mlp.gate_proj.weight")) * lin(h, "mlp.up_proj.weight"),
                    "mlp.down_proj.weight")
    return x, kv


def _exact_model(case, seed):
    cfg = _config(case)
    w = dict(_weights(cfg, seed))
    if case.get("bits"):
        for name in w:
            if name.endswith("_proj.weight"):
                w[name] = _quantized(w[name], case["bits"])
    emb = w["model.embed_tokens.weight"]

    def past(slot, length):
        return [[t.double().transpose(0, 1).contiguous() for t in _past(cfg, seed, slot, l, length)]
                for l in range(cfg.num_hidden_layers)]

    def head(x):
        h = _norm(x, w["model.norm.weight"].double())
        return h, torch.cat([h @ e.double().t() for e in emb.split(16384)], -1)

    if case["kind"] == "batch":
        ids, rows = _tokens(case, seed, cfg.vocab_size, case["n"]), []
        for i, length in enumerate(_lengths(case, seed)):
            x, _ = _forward(cfg, w, emb[int(ids[i])][None].double(), past(i, length), length)
            rows.append(x)
        return {"logits": head(torch.cat(rows))[1], "next": None}
    if case["kind"] == "prompt":
        ids = torch.from_numpy(_tokens(case, seed, cfg.vocab_size, case["n"])).long().cuda()
        x, kv = _forward(cfg, w, emb[ids].double(), past(0, case["past"]), case["past"])
        hidden = _norm(x, w["model.norm.weight"].double())
        return {"hidden": hidden, "logits": head(x[-case["logit_rows"]:])[1], "token": None, "keys": kv[-1][0],
                "values": kv[-1][1]}
    t = int(_tokens(case, seed, cfg.vocab_size, case["steps"] + 1)[0])
    kv = past(0, case["past"])
    for i in range(case["steps"] + 1):
        x, kv = _forward(cfg, w, emb[t][None].double(), kv, case["past"] + i)
        logits = head(x)[1]
        t = int(logits.argmax())
    return {"tokens": None, "token": None, "logits": logits, "keys": kv[-1][0], "values": kv[-1][1]}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prompt", "decode", "batch"):
        return _exact_model(case, seed)
    s = _op_inputs(case, seed)
    if kind == "gemv":
        return torch.cat([p.double() @ s["x"].double() for p in s["w"].split(16384)])
    if kind == "qmm":
        parts = []
        for c, sc in zip(s["codes"].split(8192), s["scales"].split(8192)):
            w = (c.double().view(c.shape[0], -1, 64) * sc.double()[..., None]).view(c.shape[0], -1)
            parts.append(s["x"].double() @ w.t().contiguous())
        return torch.cat(parts, 1)
    if kind == "sample":
        return {"token": None, "ids": None, "values": torch.topk(s["row"].double(), case["k"]).values}
    n = case["len"] if kind == "attn_decode" else case["past"] + case["rows"]
    return _attend(s["q"].double(), s["k"][:, :n].double(), s["v"][:, :n].double(), n - s["q"].shape[0])
