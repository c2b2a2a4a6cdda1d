"""The calls whose speed is measured, each through a public entry point.

A case is a dict of plain values with a "kind":

  mlp        one feed-forward half layer through the operators: RMSNorm, gate
             and up products, SwiGLU, down product with the residual add, for
             1..64 activation rows.
  head       the output head through the operators: final RMSNorm, the binary16
             vocabulary product and the greedy choice.
  attention  one decode attention call over a KV cache, ragged lengths.
  step       one eager decode step of a model (Model.forward) for 1..64
             sequences at their own positions; logits and KV cache.
  decode     a captured decode loop (Model.graph_begin and graph_run): the
             tokens, the last logits and the KV cache.
  prompt     a prompt and its first generated token (Model.generate): what a
             chat turn waits for before text appears.

Model and layer shapes are the Llama-3-8B and Llama-2-7B ones and the tiny
two-layer model of the benchmark and tests, with one or two layers and a
32000-token vocabulary; weights are random GGUF blocks with the value spread of
quantised weights.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from janus_amd import ops
from janus_amd.model import Model
from janus_amd.synth import ModelSpec, Tensor

DEV = "cuda:0"
F16, Q4_0, Q8_0, Q4_K, Q5_K = ops.DT_F16, ops.DT_Q4_0, ops.DT_Q8_0, ops.DT_Q4_K, ops.DT_Q5_K
FORMATS = {"f16": F16, "q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q5_k": Q5_K}
DTYPES = {"f16": torch.float16, "f32": torch.float32}
EPS = 1e-5
# hidden, heads, KV heads, FFN, RoPE base
SHAPES = {"tiny": (256, 4, 2, 512, 10000.0),
          "llama2_7b": (4096, 32, 32, 11008, 10000.0),
          "llama3_8b": (4096, 32, 8, 14336, 500000.0)}
BLOCK_BYTES = {F16: (1, 2), Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176)}


# ---- cases ---------------------------------------------------------------------

def listed():
    return [
        # the smallest whole call: a step of the tiny model on the default dtypes
        dict(name="step_tiny_1", kind="step", shape="tiny", fmt="q8_0", act="f32", layers=2, vocab=512,
             rows=1, ctx=40, max_seq=64),
        # one token through a feed-forward layer, the ordinary decode product
        dict(name="mlp_q4_0_1", kind="mlp", fmt="q4_0", act="f16", rows=1, hidden=4096, ffn=14336),
        # a small batch on the operators' default (the reference's) activation dtype
        dict(name="mlp_q4_k_f32_16", kind="mlp", fmt="q4_k", act="f32", rows=16, hidden=4096, ffn=11008),
        # an odd batch above one 32-row tile
        dict(name="mlp_q5_k_33", kind="mlp", fmt="q5_k", act="f16", rows=33, hidden=4096, ffn=14336),
        # the greedy head of a few sequences on f32 activations
        dict(name="head_f32_3", kind="head", act="f32", rows=3, hidden=4096, vocab=32000),
        # one long conversation
        dict(name="attn_f16_1", kind="attention", kv="f16", heads=32, kv_heads=8, head_dim=128, batch=1, max_len=6000),
        # the ragged batch of the benchmark: contexts of 128 to 8192
        dict(name="attn_f16_16", kind="attention", kv="f16", heads=32, kv_heads=8, head_dim=128, batch=16,
             max_len=8192),
        # the default cache dtype, multi-head, a handful of sequences
        dict(name="attn_f32_5", kind="attention", kv="f32", heads=32, kv_heads=32, head_dim=128, batch=5, max_len=1000),
        # captured decode of one conversation: the chat loop
        dict(name="decode_q4_0_1", kind="decode", shape="llama3_8b", fmt="q4_0", act="f16", layers=2, vocab=32000,
             rows=1, ctx=700, max_seq=1024, steps=4),
        # a serving step: 32 ragged sequences
        dict(name="step_q4_0_32", kind="step", shape="llama3_8b", fmt="q4_0", act="f16", layers=1, vocab=32000,
             rows=32, ctx=2000, max_seq=2048),
        # time to the first token of an ordinary prompt on binary16 activations
        dict(name="prompt_q4_0_512", kind="prompt", shape="llama3_8b", fmt="q4_0", act="f16", layers=1, vocab=32000,
             prompt=512, max_seq=1024),
        # the same on the default dtypes (f32 activations and cache), ragged length
        dict(name="prompt_q4_k_f32_133", kind="prompt", shape="llama2_7b", fmt="q4_k", act="f32", layers=1,
             vocab=32000, prompt=133, max_seq=512),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "head", "attention", "attention", "step", "decode", "prompt"])
    fmt = rng.choice(sorted(FORMATS))
    act = rng.choice(["f16", "f32"])
    if kind == "mlp":
        return dict(kind=kind, fmt=fmt, act=act, rows=_log_int(rng, 1, 64), hidden=rng.choice([256, 1024, 2048, 4096]),
                    ffn=256 * _log_int(rng, 2, 56))
    if kind == "head":
        return dict(kind=kind, act=act, rows=_log_int(rng, 1, 64), hidden=rng.choice([256, 1024, 2048, 4096]),
                    vocab=_log_int(rng, 500, 32000))
    if kind == "attention":
        heads, kv_heads, hd = rng.choice([(32, 8, 128), (32, 32, 128), (4, 2, 64), (32, 4, 128), (16, 16, 64)])
        batch = _log_int(rng, 1, 64)
        top = max(16, min(8192, 130000 * 8 // (batch * kv_heads)))
        return dict(kind=kind, kv=act, heads=heads, kv_heads=kv_heads, head_dim=hd, batch=batch,
                    max_len=_log_int(rng, 16, top))
    shape = rng.choice(sorted(SHAPES))
    if shape == "tiny":
        base = dict(shape=shape, fmt=fmt, act=act, layers=2, vocab=512)
    else:
        base = dict(shape=shape, fmt=fmt if fmt != "f16" else "q8_0", act=act, layers=1, vocab=_log_int(rng, 500, 32000))
    if kind == "prompt":
        prompt = _log_int(rng, 5, 400)
        return dict(kind=kind, **base, prompt=prompt, max_seq=prompt + rng.randint(2, 200))
    rows, ctx = _log_int(rng, 1, 32), _log_int(rng, 16, 1500)
    if kind == "decode":
        rows = rng.choice([1, 1, rows])
        return dict(kind=kind, **base, rows=rows, ctx=ctx, max_seq=ctx + rng.randint(8, 300), steps=rng.randint(2, 4))
    return dict(kind=kind, **base, rows=rows, ctx=ctx, max_seq=ctx + rng.randint(2, 300))


# ---- inputs --------------------------------------------------------------------

def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1000003 + salt) & 0x7FFFFFFF)
    return g


def _f16_bytes(x, nblk):
    return x.to(torch.float16).view(torch.uint8).reshape(nblk, 2)


def _blocks(g, fmt, n, k, sigma=0.02):
    """GGUF bytes [blocks, block bytes] on the GPU of random weights with a
    spread of about `sigma`; block scales are normal binary16 numbers."""
    width, nbytes = BLOCK_BYTES[fmt]
    nblk = n * k // width
    if fmt == F16:
        w = (torch.randn(n, k, generator=g, device=DEV) * sigma).to(torch.float16)
        w[w.abs() < 6.2e-5] = 0   # the loader flushes binary16 subnormals
        return w.view(torch.uint8).reshape(nblk, 2)
    out = torch.randint(0, 256, (nblk, nbytes), generator=g, device=DEV, dtype=torch.uint8)
    u = torch.rand(nblk, generator=g, device=DEV) + 0.5
    if fmt == Q4_0:
        out[:, 0:2] = _f16_bytes(u * (sigma / 4.6), nblk)
    elif fmt == Q8_0:
        out[:, 0:2] = _f16_bytes(u * (sigma / 74.0), nblk)
    else:   # K-quants: six-bit scales and mins uniform, the mins centring the values
        mid, step = (7.5, 1.6e-4) if fmt == Q4_K else (15.5, 0.8e-4)
        out[:, 0:2] = _f16_bytes((u * step).clamp(min=6.2e-5), nblk)
        out[:, 2:4] = _f16_bytes(u * step * mid, nblk)
    return out


def _host(blocks):
    return blocks.reshape(-1).cpu().numpy()


def _dequant(raw, fmt, n, k):
    """Float64 values [n, k] of GGUF blocks."""
    if fmt == F16:
        return raw.reshape(-1).view(torch.float16).reshape(n, k).double()
    d = raw[:, 0:2].contiguous().view(torch.float16).double()   # [blocks, 1]
    if fmt == Q8_0:
        return (raw[:, 2:].contiguous().view(torch.int8).double() * d).reshape(n, k)
    if fmt == Q4_0:
        q = raw[:, 2:]
        return ((torch.cat([q & 15, q >> 4], 1).double() - 8.0) * d).reshape(n, k)
    dmin = raw[:, 2:4].contiguous().view(torch.float16).double()
    s = raw[:, 4:16].int()
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    qs = raw[:, -128:].reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
    if fmt == Q5_K:
        bits = torch.arange(8, device=raw.device).reshape(1, 8, 1)
        q = q + 16.0 * ((raw[:, 16:48].int().reshape(-1, 1, 32) >> bits) & 1).double()
    return ((d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]).reshape(n, k)


_ENGINE = None


def _engine():
    """The process's compute engine, made once as a program makes it."""
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = ops.ComputeEngine(0)
    return _ENGINE


def _gamma(g, n):
    return 1 + 0.02 * torch.randn(n, generator=g, device=DEV)


def _hidden(g, rows, hidden):
    """A residual stream: normal values with a few strong channels."""
    x = torch.randn(rows, hidden, generator=g, device=DEV)
    strong = torch.randint(0, hidden, (max(1, hidden // 256),), generator=g, device=DEV)
    x[:, strong] *= 8.0
    return x


def _mlp_inputs(case, seed):
    g, h, f, fmt = _gen(seed, 11), case["hidden"], case["ffn"], FORMATS[case["fmt"]]
    return dict(x=_hidden(g, case["rows"], h), gamma=_gamma(g, h), gate=_blocks(g, fmt, f, h),
                up=_blocks(g, fmt, f, h), down=_blocks(g, fmt, h, f))


def _head_inputs(case, seed):
    g, h = _gen(seed, 12), case["hidden"]
    return dict(x=_hidden(g, case["rows"], h), gamma=_gamma(g, h), w=_blocks(g, F16, case["vocab"], h))


def _lengths(g, count, top):
    low = max(1, min(top, top // 64))
    return torch.randint(low, top + 1, (count,), generator=g, device=DEV, dtype=torch.int32)


def _attention_inputs(case, seed):
    g, b, kvh, hd, top = _gen(seed, 13), case["batch"], case["kv_heads"], case["head_dim"], case["max_len"]
    lens = _lengths(g, b, top)
    lens[0] = top
    base = torch.zeros_like(lens)
    base[1:] = lens.cumsum(0)[:-1].to(torch.int32)
    rows = int(lens.sum().item())
    kv = [torch.randn(rows, kvh, hd, generator=g, device=DEV).to(DTYPES[case["kv"]]) for _ in range(2)]
    return dict(q=2 * torch.randn(b, case["heads"], hd, generator=g, device=DEV), k=kv[0], v=kv[1], lens=lens, base=base)


def _model_tensors(case, seed):
    h, heads, kvh, f, _ = SHAPES[case["shape"]]
    g, fmt, vocab, kvd = _gen(seed, 14), FORMATS[case["fmt"]], case["vocab"], kvh * (h // heads)
    t = {"token_embd.weight": (F16, vocab, h, _blocks(g, F16, vocab, h, 1.0))}
    for i in range(case["layers"]):
        p = "blk.%d." % i
        t[p + "attn_norm.weight"] = (ops.DT_F32, h, 0, _gamma(g, h))
        t[p + "ffn_norm.weight"] = (ops.DT_F32, h, 0, _gamma(g, h))
        for name, n, k in (("attn_q", h, h), ("attn_k", kvd, h), ("attn_v", kvd, h), ("attn_output", h, h),
                           ("ffn_gate", f, h), ("ffn_up", f, h), ("ffn_down", h, f)):
            t[p + name + ".weight"] = (fmt, n, k, _blocks(g, fmt, n, k))
    t["output_norm.weight"] = (ops.DT_F32, h, 0, _gamma(g, h))
    t["output.weight"] = (F16, vocab, h, _blocks(g, F16, vocab, h))
    return t


def _step_inputs(case, seed):
    """Tokens and positions of a step, and the caches' contents before it."""
    h, heads, kvh, _, _ = SHAPES[case["shape"]]
    g, rows, hd = _gen(seed, 15), case["rows"], h // heads
    tokens = torch.randint(0, case["vocab"], (rows,), generator=g, device=DEV)
    positions = _lengths(g, rows, case["ctx"]) - 1
    positions[0] = case["ctx"] - 1
    kv = [torch.randn(case["layers"], rows * case["max_seq"], kvh, hd, generator=g, device=DEV).to(DTYPES[case["act"]])
          for _ in range(2)]
    return tokens.tolist(), positions.tolist(), kv


def _prompt_inputs(case, seed):
    h, heads, kvh, _, _ = SHAPES[case["shape"]]
    g = _gen(seed, 16)
    tokens = torch.randint(0, case["vocab"], (case["prompt"],), generator=g, device=DEV)
    kv = [torch.zeros(case["layers"], case["max_seq"], kvh, h // heads, device=DEV, dtype=DTYPES[case["act"]])
          for _ in range(2)]
    return tokens.tolist(), kv


def _model(case, seed, rows, kv):
    h, heads, kvh, f, theta = SHAPES[case["shape"]]
    tensors = [Tensor(name, typ, n, k, _host(raw) if k else raw.cpu().numpy())
               for name, (typ, n, k, raw) in _model_tensors(case, seed).items()]
    dt = ops.DT_F16 if case["act"] == "f16" else ops.DT_F32
    m = Model(_engine(), ModelSpec(h, heads, kvh, f, case["vocab"], case["layers"], EPS, theta, tensors),
              max_seq_len=case["max_seq"], max_batch=rows, kv_dtype=dt, act_dtype=dt)
    m.spec.tensors = []   # uploaded
    m.set_kv_cache(*kv)
    return m


class _DeviceArray:
    """A device buffer of the library, for torch.as_tensor (which keeps this
    object, and so its owner, alive with the tensor)."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 3}


def _logits(m, rows, vocab):
    return torch.as_tensor(_DeviceArray(m, m.logits_ptr(), (rows, vocab), "<f4"), device=DEV)


def prepare(case, seed):
    e, kind = _engine(), case["kind"]
    if kind == "mlp":
        i, fmt, h, f = _mlp_inputs(case, seed), FORMATS[case["fmt"]], case["hidden"], case["ffn"]
        act, rows = DTYPES[case["act"]], case["rows"]
        return dict(kind=kind, rows=rows, h=h, f=f, x=i["x"], gamma=i["gamma"],
                    gate=ops.GpuTensor(e, fmt, f, h, _host(i["gate"])), up=ops.GpuTensor(e, fmt, f, h, _host(i["up"])),
                    down=ops.GpuTensor(e, fmt, h, f, _host(i["down"])),
                    xn=torch.empty(rows, h, dtype=act, device=DEV), g=torch.empty(rows, f, device=DEV),
                    u=torch.empty(rows, f, device=DEV), act=torch.empty(rows, f, dtype=act, device=DEV),
                    out=torch.empty(rows, h, device=DEV))
    if kind == "head":
        i, rows, h, v = _head_inputs(case, seed), case["rows"], case["hidden"], case["vocab"]
        return dict(kind=kind, rows=rows, h=h, v=v, x=i["x"], gamma=i["gamma"],
                    w=ops.GpuTensor(e, F16, v, h, _host(i["w"])),
                    xn=torch.empty(rows, h, dtype=DTYPES[case["act"]], device=DEV),
                    logits=torch.empty(rows, v, device=DEV), ids=torch.empty(rows, dtype=torch.int32, device=DEV))
    if kind == "attention":
        return dict(kind=kind, case=dict(case), out=torch.empty(case["batch"], case["heads"], case["head_dim"], device=DEV),
                    **_attention_inputs(case, seed))
    if kind == "prompt":
        tokens, kv = _prompt_inputs(case, seed)
        return dict(kind=kind, tokens=tokens, kv=kv, v=case["vocab"], model=_model(case, seed, 1, kv))
    tokens, positions, kv = _step_inputs(case, seed)
    return dict(kind=kind, tokens=tokens, positions=positions, kv=kv, rows=case["rows"], v=case["vocab"],
                steps=case.get("steps", 0), model=_model(case, seed, case["rows"], kv))


# ---- one pass ------------------------------------------------------------------

def run(s):
    e, kind = _engine(), s["kind"]
    if kind == "mlp":
        rows, h, f = s["rows"], s["h"], s["f"]
        ops.rmsnorm(e, s["x"], s["xn"], s["gamma"], rows, h, EPS)
        ops.gemm_auto(e, s["xn"], s["gate"], s["g"], 1, rows, h, f)
        ops.gemm_auto(e, s["xn"], s["up"], s["u"], 1, rows, h, f)
        ops.swiglu(e, s["g"], s["u"], s["act"], rows * f)
        ops.gemm_residual(e, s["act"], s["down"], s["x"], s["out"], rows)
        return {name: s[name] for name in ("xn", "g", "u", "act", "out")}
    if kind == "head":
        ops.rmsnorm(e, s["x"], s["xn"], s["gamma"], s["rows"], s["h"], EPS)
        ops.gemm_auto(e, s["xn"], s["w"], s["logits"], 1, s["rows"], s["h"], s["v"])
        ops.argmax(e, s["logits"], s["ids"], s["v"], s["rows"])
        return {"logits": s["logits"], "ids": s["ids"]}
    if kind == "attention":
        c = s["case"]
        ops.compute_attention(e, s["q"], s["k"], s["v"], s["out"], c["batch"], 0, c["max_len"], c["heads"],
                              c["kv_heads"], c["head_dim"], s["base"], s["lens"], c["max_len"])
        return s["out"]
    m = s["model"]
    if kind == "prompt":
        out = m.generate(s["tokens"], 1)
        return {"tokens": np.asarray(out, np.int64), "logits": _logits(m, 1, s["v"]), "k": s["kv"][0], "v": s["kv"][1]}
    if kind == "decode":
        m.graph_begin(s["tokens"], s["positions"])
        m.graph_run(s["steps"])
        return {"tokens": np.asarray(m.graph_tokens(s["rows"]), np.int64), "logits": _logits(m, s["rows"], s["v"]),
                "k": s["kv"][0], "v": s["kv"][1]}
    m.forward(s["tokens"], s["positions"])
    return {"logits": _logits(m, s["rows"], s["v"]), "k": s["kv"][0], "v": s["kv"][1]}


# ---- what a pass needs ---------------------------------------------------------

def _wbytes(fmt, n, k):
    width, nbytes = BLOCK_BYTES[FORMATS[fmt]]
    return n * k // width * nbytes


def _mean_len(case):
    top = case["ctx"] if "ctx" in case else case["max_len"]
    return (max(1, min(top, top // 64)) + top) / 2.0


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        rows, h, f = case["rows"], case["hidden"], case["ffn"]
        return {"bytes": 3 * _wbytes(case["fmt"], f, h) + rows * h * 8 + 4 * h, "flops": 6.0 * rows * h * f}
    if kind == "head":
        rows, h, v = case["rows"], case["hidden"], case["vocab"]
        return {"bytes": 2 * v * h + rows * (4 * h + 4 * v + 4) + 4 * h, "flops": 2.0 * rows * h * v}
    if kind == "attention":
        kvb = 2 if case["kv"] == "f16" else 4
        n = case["max_len"] + (case["batch"] - 1) * _mean_len(case)
        row, q = case["kv_heads"] * case["head_dim"], case["heads"] * case["head_dim"]
        return {"bytes": n * 2 * row * kvb + case["batch"] * q * 8, "flops": 4.0 * n * q}
    h, heads, kvh, f, _ = SHAPES[case["shape"]]
    kvd, kvb = kvh * (h // heads), 2 if case["act"] == "f16" else 4
    layer = 2 * _wbytes(case["fmt"], h, h) + 2 * _wbytes(case["fmt"], kvd, h) + 3 * _wbytes(case["fmt"], f, h)
    params, head = 2 * h * h + 2 * kvd * h + 3 * f * h, 2 * case["vocab"] * h
    L, v = case["layers"], case["vocab"]
    if kind == "prompt":
        n = case["prompt"] + 1   # the last prompt token is fed twice
        return {"bytes": L * (layer + n * 2 * kvd * kvb) + head + n * 2 * h + 4 * v,
                "flops": 2.0 * n * L * params + L * 2.0 * n * n * h + 2.0 * v * h}
    rows, steps = case["rows"], case.get("steps", 1)
    n = case["ctx"] + (rows - 1) * _mean_len(case)
    return {"bytes": steps * (L * (layer + n * 2 * kvd * kvb) + head + rows * (2 * h + 4 * v)),
            "flops": steps * (rows * (2.0 * L * params + 2.0 * v * h) + L * 4.0 * n * h)}


def tolerance(case):
    kind, act = case["kind"], case.get("act", case.get("kv"))
    if kind == "mlp":   # f32 sums; with f16, the norm's and SwiGLU's outputs round to binary16
        return {"rel": 2e-6, "max": 2e-5} if act == "f32" else {"rel": 1.5e-3, "max": 1.5e-2}
    if kind == "head":   # the greedy id may differ at a tie within rounding
        return {"rel": 2e-6, "max": 2e-5, "differ": 0.05} if act == "f32" else {"rel": 1e-3, "max": 1e-2, "differ": 0.05}
    if kind == "attention":
        return {"rel": 4e-6, "max": 4e-5}
    # measured against 64 bits: up to 9e-6 on f32, 4e-4 on binary16 activations
    return {"rel": 4e-5, "max": 4e-4, "differ": 0.05} if act == "f32" else {"rel": 4e-3, "max": 4e-2, "differ": 0.05}


# ---- the same results in 64 bits -----------------------------------------------

def _norm64(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def _silu64(x):
    return x / (1.0 + torch.exp(-x))


def _rope64(x, positions, theta):
    """Half-split rotation of x [rows, heads, hd]; angles in binary32 as the
    cos/sin table defines them."""
    half = x.shape[-1] // 2
    expo = np.float32(2) * np.arange(half, dtype=np.float32) / np.float32(2 * half)
    ang = np.asarray(positions, np.float32)[:, None] / np.power(np.float32(theta), expo).astype(np.float32)
    ang = torch.from_numpy(ang.astype(np.float64)).to(x.device)[:, None, :]
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _attend64(q, k, v):
    """q [rows, heads, hd] over k, v [len, kv heads, hd]; row r of q sees the
    first len - rows + 1 + r positions."""
    rows, heads, hd = q.shape
    n, rep = k.shape[0], heads // k.shape[1]
    out = torch.empty_like(q)
    seen = torch.arange(n, device=q.device)[None, :] <= torch.arange(n - rows, n, device=q.device)[:, None]
    for h in range(heads):
        sc = q[:, h] @ k[:, h // rep].double().T.contiguous() / math.sqrt(hd)
        out[:, h] = torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ v[:, h // rep].double()
    return out


def _forward64(case, w, tokens, spans, kv):
    """One pass of tokens through the model. spans: (first row, rows, first
    position, KV base row) of each sequence. Writes kv, returns the logits."""
    h, heads, kvh, _, theta = SHAPES[case["shape"]]
    hd = h // heads
    x = w["token_embd.weight"][torch.as_tensor(tokens, device=DEV)]
    pos = np.concatenate([np.arange(p, p + n) for _, n, p, _ in spans])
    for i in range(case["layers"]):
        p = "blk.%d." % i
        xn = _norm64(x, w[p + "attn_norm.weight"])
        q = _rope64((xn @ w[p + "attn_q.weight"].T).reshape(-1, heads, hd), pos, theta)
        k = _rope64((xn @ w[p + "attn_k.weight"].T).reshape(-1, kvh, hd), pos, theta)
        v = (xn @ w[p + "attn_v.weight"].T).reshape(-1, kvh, hd)
        att = torch.empty_like(q)
        for r, n, first, base in spans:
            kv[0][i, base + first:base + first + n] = k[r:r + n]
            kv[1][i, base + first:base + first + n] = v[r:r + n]
            att[r:r + n] = _attend64(q[r:r + n], kv[0][i, base:base + first + n], kv[1][i, base:base + first + n])
        x = x + att.reshape(-1, h) @ w[p + "attn_output.weight"].T
        xn = _norm64(x, w[p + "ffn_norm.weight"])
        x = x + (_silu64(xn @ w[p + "ffn_gate.weight"].T) * (xn @ w[p + "ffn_up.weight"].T)) @ w[p + "ffn_down.weight"].T
    return _norm64(x, w["output_norm.weight"]) @ w["output.weight"].T


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        i, fmt, h, f = _mlp_inputs(case, seed), FORMATS[case["fmt"]], case["hidden"], case["ffn"]
        x = i["x"].double()
        xn = _norm64(x, i["gamma"])
        g, u = xn @ _dequant(i["gate"], fmt, f, h).T, xn @ _dequant(i["up"], fmt, f, h).T
        act = _silu64(g) * u
        return {"xn": xn, "g": g, "u": u, "act": act, "out": x + act @ _dequant(i["down"], fmt, h, f).T}
    if kind == "head":
        i = _head_inputs(case, seed)
        return {"logits": _norm64(i["x"].double(), i["gamma"]) @ _dequant(i["w"], F16, case["vocab"], case["hidden"]).T,
                "ids": None}
    if kind == "attention":
        i = _attention_inputs(case, seed)
        out = torch.empty(i["q"].shape, dtype=torch.float64, device=DEV)
        for b, (n, base) in enumerate(zip(i["lens"].tolist(), i["base"].tolist())):
            out[b:b + 1] = _attend64(i["q"][b:b + 1].double(), i["k"][base:base + n], i["v"][base:base + n])
        return out
    w = {name: _dequant(raw, typ, n, k) if k else raw.double()
         for name, (typ, n, k, raw) in _model_tensors(case, seed).items()}
    if kind == "prompt":
        tokens, kv = _prompt_inputs(case, seed)
        kv = [t.double() for t in kv]
        logits = _forward64(case, w, tokens + tokens[-1:], [(0, len(tokens) + 1, 0, 0)], kv)[-1:]
        return {"tokens": None, "logits": logits, "k": kv[0], "v": kv[1]}
    tokens, positions, kv = _step_inputs(case, seed)
    kv = [t.double() for t in kv]
    for step in range(case.get("steps", 1)):
        spans = [(r, 1, p + step, r * case["max_seq"]) for r, p in enumerate(positions)]
        logits = _forward64(case, w, tokens, spans, kv)
        tokens = logits.argmax(-1).tolist()
    out = {"logits": logits, "k": kv[0], "v": kv[1]}
    return {"tokens": None, **out} if kind == "decode" else out
