"""The work that is timed: what a program using this package has it do.

One pass of every case goes through the package's public entry points: the
operators of ``cosxamix_amd.ops``, the sampler, and ``forward.Modelo``. Sizes
are those of the package's model configurations (daiss-0.5b, daiss-3b, the
Llama-3-8B shape). Every entry point here computes f32 values in a documented
order (that of the reference's scalar code), or is the model made of them, so
the model's cases and the sampler's are compared bit for bit: in a model a
single changed rounding flips an i8 activation and travels through all layers
that follow. The operators state what f32 sums give.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from cosxamix_amd import _lib as L
from cosxamix_amd import forward as F
from cosxamix_amd import ops
from cosxamix_amd import sampler

TYPES = {"Q4_K": L.Q4_K, "Q5_K": L.Q5_K, "Q6_K": L.Q6_K, "Q8_0": L.Q8_0}
SUB = {"Q4_K": 32, "Q5_K": 32, "Q6_K": 16, "Q8_0": 32}
BLOCK = {"Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210), "Q8_0": (32, 34)}
MODELS = {"0.5b": F.DAISS_0_5B, "3b": F.DAISS_3B, "8b": F.LLAMA3_8B}
DEV = "cuda:0"


def listed():
    return [
        # one token's gate (or up) projection of the 3B model: the smallest
        # call a decoding program makes, where launches and latency count
        dict(name="row_q4k", kind="matmul", m=1, n=11008, k=2048, type="Q4_K"),
        # one token's q, k and v in one call, v in Q6_K as Q4_K_M files hold it
        dict(name="qkv_row", kind="rows", k=2048, n0=2048, n1=256, n2=256, t0="Q4_K", t1="Q4_K",
             t2="Q6_K"),
        # a handful of rows (drafted tokens, a few sequences) times the down
        # projection
        dict(name="down_q4k_8", kind="matmul", m=8, n=2048, k=11008, type="Q4_K"),
        # a prompt's gate projection
        dict(name="gate_q4k_512", kind="matmul", m=512, n=11008, k=2048, type="Q4_K"),
        # a short odd prompt times the down projection in Q6_K (Q4_K_M files)
        dict(name="down_q6k_77", kind="matmul", m=77, n=2048, k=11008, type="Q6_K"),
        # a prompt's gate projection of the 0.5B model, in Q8_0 blocks
        dict(name="gate_q8_512", kind="matmul", m=512, n=4864, k=896, type="Q8_0"),
        # a chunk of a prompt's attention over what is already cached
        dict(name="attn_256", kind="attention", tokens=256, total=512, heads=16, kv=2, hd=128),
        # one token's attention over a long cache (8B shape)
        dict(name="attn_row_8448", kind="attention_row", total=8448, heads=32, kv=8, hd=128),
        # one draw at temperature 0.8, top-p 0.9 over the 3B vocabulary
        dict(name="sample", kind="sample", vocab=151936, temp=0.8, top_p=0.9),
        # the whole 3B model over a 512-token prompt
        dict(name="prefill_3b", kind="prefill", model="3b", layers=36, prefix=0, tokens=512,
             type="Q4_K", down="Q4_K", out="Q4_K"),
        # 32 greedy tokens of the whole 3B model after that prompt, and the
        # logits that follow
        dict(name="decode_3b", kind="decode", model="3b", layers=36, prefix=512, tokens=32,
             type="Q4_K", down="Q4_K", out="Q4_K"),
        # a long prompt through two layers of the 8B shape (Q5_K ffn_down)
        dict(name="prefill_8b_8192", kind="prefill", model="8b", layers=2, prefix=0, tokens=8192,
             type="Q4_K", down="Q5_K", out="Q4_K"),
    ]


# (rows, width) of the models' matrices whose width is whole 256-value blocks,
# and those of the 0.5B model (Q8_0)
SHAPES = [(2048, 2048), (256, 2048), (11008, 2048), (2048, 11008), (4096, 4096), (1024, 4096),
          (14336, 4096), (4096, 14336)]
SHAPES_05B = [(896, 896), (128, 896), (4864, 896), (896, 4864)]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random):
    kind = rng.choice(["matmul", "matmul", "matmul", "matmul", "rows", "attention", "attention",
                       "attention_row", "sample", "prefill", "prefill", "decode"])
    if kind == "matmul":
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0"])
        n, k = rng.choice(SHAPES_05B if t == "Q8_0" else SHAPES)
        if rng.random() < 0.25:  # an odd number of rows, as a cut or merged matrix has
            n = rng.randrange(n // 2 + 1, n, 2)
        return dict(kind=kind, m=_log(rng, 1, 700), n=n, k=k, type=t)
    if kind == "rows":
        k, n0, n1 = rng.choice([(2048, 2048, 256), (4096, 4096, 1024)])
        t = rng.choice(["Q4_K", "Q5_K"])
        return dict(kind=kind, k=k, n0=n0, n1=n1, n2=n1, t0=t, t1=t,
                    t2=rng.choice([t, "Q6_K"]))
    if kind in ("attention", "attention_row"):
        heads, kv, hd = rng.choice([(14, 2, 64), (16, 2, 128), (32, 8, 128)])
        if kind == "attention_row":
            return dict(kind=kind, total=_log(rng, 2, 10000), heads=heads, kv=kv, hd=hd)
        tokens = _log(rng, 2, 512)
        return dict(kind=kind, tokens=tokens, total=tokens + rng.randrange(0, 1500), heads=heads,
                    kv=kv, hd=hd)
    if kind == "sample":
        return dict(kind=kind, vocab=rng.choice([32000, 128256, 151936]) - rng.randrange(0, 64),
                    temp=round(rng.uniform(0.3, 1.5), 2),
                    top_p=rng.choice([0.5, 0.8, 0.9, 0.95, 1.0]))
    model = rng.choice(["0.5b", "3b", "8b"])
    if model == "0.5b":
        t = down = out = "Q8_0"
    else:
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K"])
        down = rng.choice([t, "Q6_K"])
        out = rng.choice([t, "Q6_K"])
    layers = rng.randrange(1, 5)
    if kind == "prefill":
        return dict(kind=kind, model=model, layers=layers, prefix=rng.choice([0, 0, 300]),
                    tokens=_log(rng, 2, 4000), type=t, down=down, out=out)
    return dict(kind=kind, model=model, layers=layers, prefix=_log(rng, 2, 6000),
                tokens=rng.randrange(8, 33), type=t, down=down, out=out)


# ------------------------------------------------------------------ inputs
def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + salt * 7919) % (1 << 62))
    return g


def _ints(g, lo, hi, shape):  # lo .. hi, both ends included
    return torch.randint(lo, hi + 1, shape, generator=g, device=DEV, dtype=torch.int32)


def _half(x):  # f16 bytes [..., 2]
    return x.to(torch.float16).contiguous().view(torch.uint8).reshape(*x.shape, 2)


def _codes(g, nb, vals, mid, sd, hi):  # quantized values around the middle of their range
    r = torch.randn((nb, vals), generator=g, device=DEV)
    return (r * sd + mid).round().clamp(0, hi).to(torch.int32)


def _weights(g, n, k, t):
    """n rows of k values of type t: their block bytes, and the values' parts
    (scale and offset per sub-block, codes) for _values."""
    vpb, _ = BLOCK[t]
    nb = n * k // vpb
    spread = 0.75 + 0.5 * torch.rand((nb,), generator=g, device=DEV)
    if t == "Q8_0":
        d = (0.02 / 42.0 * spread).to(torch.float16)
        q = (torch.randn((nb, 32), generator=g, device=DEV) * 42.0).round().clamp(-127, 127)
        raw = torch.cat([_half(d), q.to(torch.int8).view(torch.uint8)], 1)
        return raw.reshape(-1), (d[:, None], torch.zeros_like(d)[:, None], q.to(torch.int32), 32)
    if t == "Q6_K":
        d = (0.02 / (48.0 * 12.0) * spread).to(torch.float16)
        sc = _ints(g, 24, 80, (nb, 16)) * (2 * _ints(g, 0, 1, (nb, 16)) - 1)
        q = _codes(g, nb, 256, 32.0, 12.0, 63)
        c = q.reshape(nb, 2, 4, 32)  # [half][group][value]
        ql = torch.stack([(c[:, :, 0] & 15) | ((c[:, :, 2] & 15) << 4),
                          (c[:, :, 1] & 15) | ((c[:, :, 3] & 15) << 4)], 2).reshape(nb, 128)
        qh = ((c[:, :, 0] >> 4) | ((c[:, :, 1] >> 4) << 2) | ((c[:, :, 2] >> 4) << 4) |
              ((c[:, :, 3] >> 4) << 6)).reshape(nb, 64)
        raw = torch.cat([ql.to(torch.uint8), qh.to(torch.uint8),
                         sc.to(torch.int8).view(torch.uint8), _half(d)], 1)
        scale = d.double()[:, None] * sc.double()
        return raw.reshape(-1), (scale, -32.0 * scale, q, 16)
    hi = 15 if t == "Q4_K" else 31
    mid, sd = hi / 2.0, hi / 5.0
    d = (0.02 / (48.0 * sd) * spread).to(torch.float16)
    dmin = (d.float() * mid).to(torch.float16)
    sc = _ints(g, 32, 63, (nb, 8))
    mn = (sc + _ints(g, -3, 3, (nb, 8))).clamp(0, 63)
    q = _codes(g, nb, 256, mid, sd, hi)
    scales = torch.cat([(sc[:, :4] | ((sc[:, 4:] >> 4) << 6)), (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)),
                        ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4))], 1)
    c = q.reshape(nb, 4, 2, 32)
    qs = ((c[:, :, 0] & 15) | ((c[:, :, 1] & 15) << 4)).reshape(nb, 128)
    parts = [_half(d), _half(dmin), scales.to(torch.uint8)]
    if t == "Q5_K":
        bit = (q.reshape(nb, 8, 32) >> 4) << torch.arange(8, device=DEV, dtype=torch.int32)[None, :, None]
        parts.append(bit.sum(1).to(torch.uint8))
    parts.append(qs.to(torch.uint8))
    scale = d.double()[:, None] * sc.double()
    return torch.cat(parts, 1).reshape(-1), (scale, -dmin.double()[:, None] * mn.double(), q, 32)


def _values(parts, n, k):  # the weights as f64 [n, k]
    scale, off, q, sub = parts
    v = q.double().reshape(q.shape[0], -1, sub)
    return (v * scale.double()[:, :, None] + off.double()[:, :, None]).reshape(n, k)


def _activation(x, sub):
    """The i8 activation the operators define (f32 amax / 127, half away from
    zero), as f64 values."""
    v = x.reshape(-1, sub)
    amax = v.abs().amax(1, keepdim=True)
    inv = torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax))
    y = (v * inv).double()
    q = torch.sign(y) * torch.floor(y.abs() + 0.5)
    return (q * (amax / 127.0).double()).reshape(x.shape)


def _matmul_inputs(case, seed):
    g = _gen(seed, 1)
    w, parts = _weights(g, case["n"], case["k"], case["type"])
    x = torch.randn((case["m"], case["k"]), generator=g, device=DEV)
    return w, parts, x


def _rows_inputs(case, seed):
    g = _gen(seed, 2)
    ws = [_weights(g, case[f"n{i}"], case["k"], case[f"t{i}"]) for i in range(3)]
    return ws, torch.randn((case["k"],), generator=g, device=DEV)


def _attention_inputs(case, seed):
    g = _gen(seed, 3)
    t, H, KV, hd = case.get("tokens", 1), case["heads"], case["kv"], case["hd"]
    q = torch.randn((t, H * hd), generator=g, device=DEV)
    k = torch.randn((case["total"], KV * hd), generator=g, device=DEV)
    v = torch.randn((case["total"], KV * hd), generator=g, device=DEV)
    return q, k, v


def _config(case):
    c = MODELS[case["model"]]
    return F.Config(case["layers"], c.dim, c.cabezas, c.cabezas_kv, c.ffn, c.vocab, c.contexto,
                    c.eps, c.rope)


def _model_inputs(case, seed):
    m = F.Modelo(_config(case), tipo=TYPES[case["type"]], semilla=seed + 1,
                 tipo_down=TYPES[case["down"]], tipo_salida=TYPES[case["out"]])
    r = np.random.default_rng(seed)
    toks = r.integers(0, m.cfg.vocab, case["prefix"] + case["tokens"] + 1).astype(np.uint32)
    cache = m.nueva_cache(case["prefix"] + case["tokens"] + 2)
    return m, cache, toks


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "matmul":
        s["w"], _, s["x"] = _matmul_inputs(case, seed)
        s["y"] = torch.empty((case["m"], case["n"]), device=DEV)
    elif kind == "rows":
        ws, s["x"] = _rows_inputs(case, seed)
        s["w"] = [(w, TYPES[case[f"t{i}"]]) for i, (w, _) in enumerate(ws)]
        s["y"] = [torch.empty((case[f"n{i}"],), device=DEV) for i in range(3)]
    elif kind in ("attention", "attention_row"):
        s["q"], s["k"], s["v"] = _attention_inputs(case, seed)
        s["y"] = torch.empty_like(s["q"])
    elif kind == "sample":
        s["logits"] = 2.5 * torch.randn((case["vocab"],), generator=_gen(seed, 4), device=DEV)
        s["seed"] = seed + 1
    else:
        m, cache, toks = _model_inputs(case, seed)
        s.update(model=m, cache=cache)
        n0 = case["prefix"]
        if n0:
            m.forward(toks[:n0], cache, logits=False)
        s["toks"] = toks[n0:n0 + (case["tokens"] if kind == "prefill" else 1)]
    return s


# -------------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "matmul":
        ops.matmul_auto((case["m"], case["k"], case["n"]), state["x"], state["w"],
                        TYPES[case["type"]], state["y"])
        return state["y"]
    if kind == "rows":
        ops.matmul_varias_una_fila(state["x"], state["w"], state["y"])
        return state["y"]
    if kind == "attention":
        ops.atencion(state["q"], state["k"], state["v"],
                     (case["tokens"], case["total"], case["heads"], case["kv"], case["hd"]),
                     state["y"])
        return state["y"]
    if kind == "attention_row":
        ops.atencion_decode(state["q"], state["k"], state["v"],
                            (case["total"], case["heads"], case["kv"], case["hd"]), state["y"])
        return state["y"]
    if kind == "sample":
        mu = sampler.Muestreador(state["seed"], case["temp"], case["top_p"])
        return mu.elegir(state["logits"])
    m, cache = state["model"], state["cache"]
    cache.truncar(case["prefix"])
    if kind == "prefill":
        logits, _ = m.forward(state["toks"], cache)
        return logits
    toks = m.generar(state["toks"], case["tokens"], cache)
    cache.truncar(cache.largo() - 1)  # the last token again, for the logits after it
    logits, _ = m.forward(toks[-1:], cache)
    return [toks, logits]


def exact(case, seed):
    kind = case["kind"]
    if kind == "matmul":
        _, parts, x = _matmul_inputs(case, seed)
        return torch.matmul(_activation(x, SUB[case["type"]]),
                            _values(parts, case["n"], case["k"]).t())
    if kind == "rows":
        ws, x = _rows_inputs(case, seed)
        return [torch.mv(_values(parts, case[f"n{i}"], case["k"]),
                         _activation(x, SUB[case[f"t{i}"]])) for i, (_, parts) in enumerate(ws)]
    if kind in ("attention", "attention_row"):
        q, k, v = (t.double() for t in _attention_inputs(case, seed))
        t, total, H, KV, hd = case.get("tokens", 1), case["total"], case["heads"], case["kv"], case["hd"]
        seen = (torch.arange(total, device=DEV)[None, :] <=
                torch.arange(total - t, total, device=DEV)[:, None])
        out = torch.empty_like(q)
        for h in range(H):
            g = h // (H // KV)
            kh, vh = k[:, g * hd:(g + 1) * hd], v[:, g * hd:(g + 1) * hd]
            s = torch.matmul(q[:, h * hd:(h + 1) * hd], kh.t().contiguous()) / math.sqrt(hd)
            p = torch.softmax(s.masked_fill(~seen, -math.inf), 1)
            out[:, h * hd:(h + 1) * hd] = torch.matmul(p, vh.contiguous())
        return out
    return None  # a drawn token; a whole model takes minutes in 64 bits


# ------------------------------------------------------------------ bookkeeping
def _matrix_bytes(n, k, t):
    vpb, bpb = BLOCK[t]
    return n * k // vpb * bpb


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": _matrix_bytes(n, k, case["type"]) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "rows":
        k, ns = case["k"], [case["n0"], case["n1"], case["n2"]]
        return {"bytes": sum(_matrix_bytes(n, k, case[f"t{i}"]) for i, n in enumerate(ns)) +
                4 * (k + sum(ns)), "flops": 2 * k * sum(ns)}
    if kind in ("attention", "attention_row"):
        t, total, H, KV, hd = case.get("tokens", 1), case["total"], case["heads"], case["kv"], case["hd"]
        pairs = t * (total - t) + t * (t + 1) // 2
        return {"bytes": 4 * (2 * t * H * hd + 2 * total * KV * hd), "flops": 4 * pairs * H * hd}
    if kind == "sample":
        return {"bytes": 4 * case["vocab"], "flops": 4 * case["vocab"]}
    c = _config(case)
    kv = c.dim_kv()
    params = 2 * c.dim * c.dim + 2 * kv * c.dim + 2 * c.ffn * c.dim
    layer = (_matrix_bytes(2 * c.dim + 2 * kv + 2 * c.ffn, c.dim, case["type"]) +
             _matrix_bytes(c.dim, c.ffn, case["down"]))
    params += c.ffn * c.dim
    head = _matrix_bytes(c.vocab, c.dim, case["out"])
    n0, t = case["prefix"], case["tokens"]
    if kind == "prefill":
        pairs = t * n0 + t * (t + 1) // 2
        return {"bytes": c.capas * (layer + 8 * kv * (n0 + t)) + head + 4 * t * c.dim + 4 * c.vocab,
                "flops": c.capas * (2 * t * params + 4 * pairs * c.dim) + 2 * c.vocab * c.dim}
    steps = t + 2  # the first token, the generated ones, the last one again
    pairs = steps * n0 + steps * (steps + 1) // 2
    return {"bytes": steps * (c.capas * layer + head) + c.capas * 8 * kv * pairs + 4 * c.vocab,
            "flops": steps * (c.capas * 2 * params + 2 * c.vocab * c.dim) + c.capas * 4 * pairs * c.dim}


def tolerance(case):
    kind = case["kind"]
    if kind in ("matmul", "rows"):
        # f32 sums of k / 32 or k / 16 terms in order, measured against 64 bits
        return {"rel": 4e-6}
    if kind in ("attention", "attention_row"):
        # f32 dots, exps and sums over the positions in order
        return {"rel": 1e-5}
    return "exact"
