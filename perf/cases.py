"""The workloads this library's speed is measured on.

One case is one call (or one short run of calls) that a serving or evaluation
program makes through the public entry points: linear layers and plain matrix
products, affine-quantized linears, attention over contiguous and paged K/V
caches, the norms, and one decode step of the Llama-shaped model. Sizes come
from the repository's own workloads: the Llama-3-8B-shaped and Qwen2-0.5B
linears, attention with 32 / 8 heads of 128 and 14 / 2 heads of 64, prompts of
up to a few thousand tokens and decode batches of 1 to 256.

``listed()`` are fixed cases, ``draw(rng)`` gives further ones of the same
ranges. ``exact`` computes a case in 64 bits with plain torch.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "mlx-batch-invariant_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mlx_batch_invariant_amd as bi  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEV = "cuda"


# ---- the cases -------------------------------------------------------------------

def _linear(name, M, N, K, dtype, bias=False, layout="nk", packed=False):
    c = {"kind": "linear", "M": M, "N": N, "K": K, "dtype": dtype, "bias": bias, "layout": layout, "packed": packed}
    return {"name": name, **c} if name else c


def _qlinear(name, M, N, K, bits, gs, dtype, copy):
    c = {"kind": "qlinear", "M": M, "N": N, "K": K, "bits": bits, "gs": gs, "dtype": dtype, "copy": copy}
    return {"name": name, **c} if name else c


def _bmm(name, batch, M, N, K, dtype, trans):
    c = {"kind": "bmm", "batch": batch, "M": M, "N": N, "K": K, "dtype": dtype, "trans": trans}
    return {"name": name, **c} if name else c


def _decode(name, B, Hq, Hkv, D, L, page, dtype):
    c = {"kind": "decode", "B": B, "Hq": Hq, "Hkv": Hkv, "D": D, "L": L, "page": page, "dtype": dtype}
    return {"name": name, **c} if name else c


def _prefill(name, B, Hq, Hkv, D, Tq, L, ragged, page, dtype):
    c = {"kind": "prefill", "B": B, "Hq": Hq, "Hkv": Hkv, "D": D, "Tq": Tq, "L": L, "ragged": ragged, "page": page,
         "dtype": dtype}
    return {"name": name, **c} if name else c


def _norms(name, rows, D, dtype):
    c = {"kind": "norms", "rows": rows, "D": D, "dtype": dtype}
    return {"name": name, **c} if name else c


def _llama(name, B, pos):
    c = {"kind": "llama", "B": B, "pos": pos}
    return {"name": name, **c} if name else c


def listed():
    return [
        # One token through one projection of a 0.5B model, called eagerly: the
        # smallest call, where launch and host time count.
        _linear("linear_m1", 1, 4864, 896, "bf16"),
        # A whole prompt batch through the 8B MLP up projection: the largest product.
        _linear("linear_prefill", 4096, 14336, 4096, "bf16"),
        # x @ W + b with W stored [in, out] (a Conv1D-style layer), a ragged
        # number of tokens, through torch.addmm under the mode.
        _linear("addmm_kn", 515, 4096, 4096, "fp16", bias=True, layout="kn"),
        # Probabilities times values of an unfused attention: a batch of 128
        # small products whose right-hand side is row-major, torch.matmul
        # under the mode.
        _bmm("bmm_pv", 128, 512, 128, 512, "bf16", False),
        # A continuous-batching decode step of 96 sequences through a 4-bit MLP
        # projection, weights repacked once at load.
        _qlinear("qlinear_batch96", 96, 14336, 4096, 4, 64, "bf16", "packed"),
        # A prompt chunk through the same projection read in its stored layout.
        _qlinear("qlinear_prefill", 1024, 14336, 4096, 4, 64, "bf16", "none"),
        # One decode step of a ragged batch over contiguous caches.
        _decode("decode_ragged", 64, 32, 8, 128, 8192, 0, "bf16"),
        # The same over a paged cache with pages of 16 keys (the page size
        # block-table servers use).
        _decode("decode_paged16", 64, 32, 8, 128, 4096, 16, "fp16"),
        # Causal prefill of four whole prompts.
        _prefill("prefill_causal", 4, 32, 8, 128, 2048, 2048, False, 0, "bf16"),
        # One chunk of a chunked prefill against a longer, ragged cache.
        _prefill("prefill_chunk", 3, 14, 2, 64, 500, 4000, True, 0, "fp16"),
        # RMSNorm and LayerNorm of a large token batch.
        _norms("norms", 16384, 4096, "bf16"),
        # One decode step of the Llama-shaped model (one block and the head,
        # 4-bit weights repacked once) for four sequences: captured into a
        # graph once and replayed, as a decode loop does.
        _llama("llama_step", 4, 1000),
    ]


# Output columns and input features of the linears.
_SHAPES = ((14336, 4096), (4096, 14336), (4096, 4096), (1024, 4096), (4864, 896), (896, 4864))


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "qlinear", "qlinear", "bmm", "decode", "decode", "prefill", "prefill",
                       "norms", "llama"))
    half = rng.choice(("bf16", "fp16"))
    if kind == "linear":
        N, K = rng.choice(_SHAPES)
        layout = rng.choice(("nk", "nk", "kn"))
        dtype = rng.choice(("bf16", "bf16", "fp16", "fp32"))
        M = _log(rng, 1, 256 if dtype == "fp32" else 3000)
        if rng.random() < 0.3:                       # odd sizes: a trimmed head, an odd feature count
            N, K = N - rng.randrange(1, 64), K - rng.randrange(1, 64)
        return _linear(None, M, N, K, dtype, rng.random() < 0.4, layout,
                       layout == "nk" and dtype != "fp32" and K % 8 == 0 and rng.random() < 0.3)
    if kind == "qlinear":
        N, K = rng.choice(_SHAPES)
        M = _log(rng, 1, 3000)
        copy = rng.choice(("none", "packed", "dequantized")) if K % 256 == 0 else "none"
        return _qlinear(None, M, N, K, rng.choice((4, 4, 8)), rng.choice((32, 64, 64, 128)), half, copy)
    if kind == "bmm":
        trans = rng.random() < 0.5                   # scores (q k^T), or probabilities times values
        D, T, L = rng.choice((64, 128)), _log(rng, 1, 512), _log(rng, 16, 1024)
        M, N, K = (T, L, D) if trans else (T, D, L)
        return _bmm(None, _log(rng, 2, 128), M, N, K, half, trans)
    if kind == "decode":
        Hq, Hkv, D = rng.choice(((32, 8, 128), (14, 2, 64), (8, 8, 128)))
        B = _log(rng, 1, 64)
        return _decode(None, B, Hq, Hkv, D, _log(rng, 64, 4000), rng.choice((0, 0, 16, 32, 64, 256)), half)
    if kind == "prefill":
        Hq, Hkv, D = rng.choice(((32, 8, 128), (14, 2, 64), (8, 8, 128)))
        Tq = _log(rng, 2, 2048)
        L = Tq if rng.random() < 0.5 else Tq + _log(rng, 1, 3000)
        return _prefill(None, rng.randrange(1, 4), Hq, Hkv, D, Tq, L, L > Tq and rng.random() < 0.5,
                        rng.choice((0, 0, 0, 16, 64)), half)
    if kind == "norms":
        return _norms(None, _log(rng, 1, 16384), rng.choice((896, 4096, 4097, 1000)), rng.choice((half, half, "fp32")))
    return _llama(None, _log(rng, 1, 64), _log(rng, 16, 2000))


# ---- inputs (plain torch, made from the seed alone) ----------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(dtype)


def _codes(g, N, K, bits, gs, dtype, std):
    """A random MLX-affine weight: uniform codes; scales and biases that put
    the dequantized values around zero with standard deviation ``std``."""
    w = torch.randint(-2**31, 2**31 - 1, (N, K * bits // 32), generator=g, device=DEV, dtype=torch.int32)
    n = (1 << bits) - 1
    s = std * math.sqrt(12) / n * (0.75 + 0.5 * torch.rand((N, K // gs), generator=g, device=DEV))
    s = s.to(dtype)
    b = (-0.5 * n * s.float() + 0.1 * std * torch.randn(s.shape, generator=g, device=DEV)).to(dtype)
    return w, s, b


def _lens(case, seed):
    """Key counts of a ragged batch: half to full cache for chunks, anything
    from one key up for decode."""
    g = torch.Generator().manual_seed(seed)
    lo = case["Tq"] + (case["L"] - case["Tq"]) // 2 if case["kind"] == "prefill" else 1
    return torch.randint(lo, case["L"] + 1, (case["B"],), generator=g)


def _kv(case, g):
    """Contiguous caches [B, Hkv, L, D], or a pool of pages and its block table."""
    B, Hkv, D, L, page, dt = (case[k] for k in ("B", "Hkv", "D", "L", "page", "dtype"))
    if not page:
        return _randn(g, B, Hkv, L, D, dtype=DTYPES[dt]), _randn(g, B, Hkv, L, D, dtype=DTYPES[dt]), None
    per = -(-L // page)
    n = B * per
    k = _randn(g, n, Hkv, page, D, dtype=DTYPES[dt])
    v = _randn(g, n, Hkv, page, D, dtype=DTYPES[dt])
    table = torch.randperm(n, generator=g, device=DEV).to(torch.int32).reshape(B, per)
    return k, v, table


# The model of the llama cases: the Llama-3-8B block with one layer and a
# 32768-token head.
def _llama_cfg():
    from mlx_batch_invariant_amd.llama import LlamaConfig
    return LlamaConfig(layers=1, vocab=32768)


_LIN = ("q", "k", "v", "o", "gate", "up", "down", "head")


def _llama_weights(seed):
    """Codes of every linear, the embedding, and the tokens and caches of the step."""
    g = _gen(seed)
    h, f, V, kvd = 4096, 14336, 32768, 1024
    shapes = {"q": (h, h), "k": (kvd, h), "v": (kvd, h), "o": (h, h), "gate": (f, h), "up": (f, h), "down": (h, f),
              "head": (V, h)}
    w = {n: _codes(g, *shapes[n], 4, 64, torch.bfloat16, 0.02) for n in _LIN}
    return w, _randn(g, V, h, dtype=torch.bfloat16), g


def _llama_inputs(case, g):
    B, pos = case["B"], case["pos"]
    tok = torch.randint(0, 32768, (B, 1), generator=g, device=DEV)
    k = _randn(g, B, 8, pos + 1, 128, dtype=torch.bfloat16)
    v = _randn(g, B, 8, pos + 1, 128, dtype=torch.bfloat16)
    return tok, k, v


def _inputs(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind == "linear":
        dt = DTYPES[case["dtype"]]
        M, N, K = case["M"], case["N"], case["K"]
        x = _randn(g, M, K, dtype=dt)
        w = _randn(g, *((N, K) if case["layout"] == "nk" else (K, N)), dtype=dt, scale=0.02)
        return x, w, _randn(g, N, dtype=dt, scale=0.1) if case["bias"] else None
    if kind == "qlinear":
        dt = DTYPES[case["dtype"]]
        x = _randn(g, case["M"], case["K"], dtype=dt)
        return (x, *_codes(g, case["N"], case["K"], case["bits"], case["gs"], dt, 0.02))
    if kind == "bmm":
        dt = DTYPES[case["dtype"]]
        b, M, N, K = (case[k] for k in ("batch", "M", "N", "K"))
        if case["trans"]:
            return _randn(g, b, M, K, dtype=dt), _randn(g, b, N, K, dtype=dt)
        return torch.softmax(torch.randn((b, M, K), generator=g, device=DEV), -1).to(dt), _randn(g, b, K, N, dtype=dt)
    if kind in ("decode", "prefill"):
        q = _randn(g, case["B"], case["Hq"], case.get("Tq", 1), case["D"], dtype=DTYPES[case["dtype"]])
        return (q, *_kv(case, g))
    if kind == "norms":
        dt = DTYPES[case["dtype"]]
        x = _randn(g, case["rows"], case["D"], dtype=dt, scale=1.5)
        w = (1 + 0.1 * torch.randn(case["D"], generator=g, device=DEV)).to(dt)
        return x, w, _randn(g, case["D"], dtype=dt, scale=0.1)
    raise ValueError(kind)


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "llama":
        return _prepare_llama(st, case, seed)
    st["in"] = _inputs(case, seed)
    if kind == "linear" and case["packed"]:
        bi.cache_packed_weight(st["in"][1])
    if kind == "qlinear" and case["copy"] != "none":
        _, w, s, b = st["in"]
        keep = bi.cache_packed if case["copy"] == "packed" else bi.cache_dequantized
        keep(w, s, b, group_size=case["gs"], bits=case["bits"])
    if kind in ("decode", "prefill"):
        ragged = kind == "decode" or case["ragged"] or case["page"]
        if not ragged:
            st["lens"] = None
        elif kind == "decode" or case["ragged"]:
            st["lens"] = _lens(case, seed).to(torch.int32).to(DEV)
        else:
            st["lens"] = torch.full((case["B"],), case["L"], dtype=torch.int32, device=DEV)
    return st


def _prepare_llama(st, case, seed):
    from mlx_batch_invariant_amd.llama import Block, LlamaShaped
    from mlx_batch_invariant_amd.nn import QuantizedLinear, cache_packed_linears
    cfg = _llama_cfg()
    model = LlamaShaped.__new__(LlamaShaped)
    torch.nn.Module.__init__(model)
    weights, embed, g = _llama_weights(seed)

    def qlin(name):
        w, s, b = weights[name]
        m = QuantizedLinear.__new__(QuantizedLinear)
        torch.nn.Module.__init__(m)
        m.in_features, m.out_features, m.group_size, m.bits = s.shape[1] * 64, w.shape[0], 64, 4
        m.register_buffer("weight", w)
        m.register_buffer("scales", s)
        m.register_buffer("biases", b)
        m.bias = None
        return m

    blk = Block.__new__(Block)
    torch.nn.Module.__init__(blk)
    blk.cfg = cfg
    for n in ("attn_norm", "mlp_norm"):
        setattr(blk, n, torch.nn.RMSNorm(cfg.hidden, eps=cfg.eps, device=DEV, dtype=torch.bfloat16))
    for n in _LIN[:-1]:
        setattr(blk, n, qlin(n))
    model.cfg, model.dtype, model.device, model.embed = cfg, torch.bfloat16, torch.device(DEV), embed
    model.blocks = torch.nn.ModuleList([blk])
    model.norm = torch.nn.RMSNorm(cfg.hidden, eps=cfg.eps, device=DEV, dtype=torch.bfloat16)
    model.head = qlin("head")
    model.eval()
    cache_packed_linears(model)
    tok, k, v = _llama_inputs(case, g)
    model._ensure_rope(case["pos"] + 1)
    cache = [(k, v)]
    pos = case["pos"]
    with bi.set_batch_invariant_mode(strict=True):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model(tok, cache, pos)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = model(tok, cache, pos)
    st.update(graph=graph, out=out, cache=cache, model=model, tok=tok)
    return st


# ---- one pass ------------------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "llama":
        st["graph"].replay()
        return [st["out"], st["cache"][0][0][:, :, -1], st["cache"][0][1][:, :, -1]]
    if kind == "linear":
        x, w, bias = st["in"]
        if case["layout"] == "nk" and bias is None:
            return bi.batch_invariant_matmul(x, w.t())
        with bi.set_batch_invariant_mode(strict=True):
            if case["layout"] == "nk":
                return F.linear(x, w, bias)
            return torch.matmul(x, w) if bias is None else torch.addmm(bias, x, w)
    if kind == "qlinear":
        x, w, s, b = st["in"]
        return bi.batch_invariant_quantized_matmul(x, w, s, b, group_size=case["gs"], bits=case["bits"])
    if kind == "bmm":
        a, b = st["in"]
        with bi.set_batch_invariant_mode(strict=True):
            return torch.matmul(a, b.transpose(1, 2) if case["trans"] else b)
    if kind in ("decode", "prefill"):
        q, k, v, table = st["in"]
        scale = case["D"] ** -0.5
        mask = "causal" if kind == "prefill" else None
        if table is not None:
            return bi.batch_invariant_paged_attention(q, k, v, table, st["lens"], scale=scale, mask=mask)
        return bi.batch_invariant_attention(q, k, v, scale=scale, mask=mask, kv_lens=st["lens"])
    x, w, b = st["in"]
    return [bi.batch_invariant_rms_norm(x, w, 1e-6), bi.batch_invariant_layer_norm(x, w, b, 1e-5)]


# ---- what a pass cannot do without ----------------------------------------------------

def _keys(case):
    """Expected (query, key) pairs per head and read keys, summed over the batch."""
    B, L = case["B"], case["L"]
    if case["kind"] == "decode":
        n = B * (L + 1) / 2
        return n, n
    Tq = case["Tq"]
    mean = (L + Tq + (L - Tq) // 2) / 2 if case["ragged"] else L
    return B * (Tq * (mean - Tq) + Tq * (Tq + 1) / 2), B * mean


def work(case):
    kind = case["kind"]
    if kind == "llama":
        params = 4096 * 4096 * 2 + 2 * 1024 * 4096 + 3 * 14336 * 4096 + 32768 * 4096
        B, L = case["B"], case["pos"] + 1
        return {"bytes": params / 2 + params / 64 * 4 + B * L * 4096 + B * (32768 * 2 + 8192),
                "flops": 2 * B * params + 4 * B * L * 32 * 128}
    es = 4 if case["dtype"] == "fp32" else 2
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": es * (M * K + N * K + M * N + (N if case["bias"] else 0)), "flops": 2 * M * N * K}
    if kind == "qlinear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K * case["bits"] / 8 + 4 * N * K / case["gs"] + 2 * M * (N + K), "flops": 2 * M * N * K}
    if kind == "bmm":
        b, M, N, K = (case[k] for k in ("batch", "M", "N", "K"))
        return {"bytes": es * b * (M * K + N * K + M * N), "flops": 2 * b * M * N * K}
    if kind in ("decode", "prefill"):
        pairs, keys = _keys(case)
        D = case["D"]
        return {"bytes": es * (2 * keys * case["Hkv"] * D + 2 * case["B"] * case["Hq"] * case.get("Tq", 1) * D),
                "flops": 4 * pairs * case["Hq"] * D}
    n = case["rows"] * case["D"]
    return {"bytes": es * 3 * n + 3 * es * case["D"], "flops": 12 * n}


# About four times the relative errors measured against 64 bits: 1.7e-3 for a
# bf16 result (2.3e-3 with a quantized weight, which is rounded to bf16 too),
# 2e-4 for fp16 (3e-4 with a bias added to the rounded product), 3e-7 for fp32;
# 6.5e-3 for the model's logits, whose bf16 activations pass nine linears.
def tolerance(case):
    kind = case["kind"]
    if kind == "llama":
        return {"rel": 2.6e-2, "max": 0.2}
    rel = {"bf16": 8e-3, "fp16": 1.2e-3, "fp32": 1e-5}[case["dtype"]]
    return {"rel": rel, "max": 4 * rel}


# ---- the same in 64 bits ---------------------------------------------------------------

def _dequant(w, s, b, bits, gs):
    per = 32 // bits
    sh = torch.arange(per, device=w.device, dtype=torch.int32) * bits
    codes = (w.unsqueeze(-1) >> sh) & ((1 << bits) - 1)
    codes = codes.reshape(w.shape[0], -1, gs).double()
    return (codes * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(w.shape[0], -1)


def _attend(q, k, v, scale, offset):
    """One sequence: q [Hq, T, D], k / v [Hkv, n, D]; query t sees keys <= offset + t."""
    Hq, T, D = q.shape
    Hkv, n, _ = k.shape
    out = torch.empty_like(q)
    G = Hq // Hkv
    seen = torch.arange(n, device=q.device)[None, :] <= (torch.arange(T, device=q.device)[:, None] + offset)
    for h in range(Hkv):
        kh, vh = k[h].t().contiguous(), v[h].contiguous()
        for i in range(G):
            s = (q[h * G + i] @ kh) * scale
            s = s.masked_fill(~seen, float("-inf"))
            out[h * G + i] = torch.softmax(s, -1) @ vh
    return out


def _exact_llama(case, seed):
    weights, embed, g = _llama_weights(seed)
    tok, k, v = _llama_inputs(case, g)
    B, pos = case["B"], case["pos"]

    def lin(name, x):
        w, s, b = weights[name]
        return x @ _dequant(w, s, b, 4, 64).t().contiguous()

    def norm(x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)

    inv = 1.0 / (5e5 ** (torch.arange(0, 128, 2, dtype=torch.float64, device=DEV) / 128))
    cos, sin = (pos * inv).cos(), (pos * inv).sin()

    def rope(x):
        x1, x2 = x[..., :64], x[..., 64:]
        return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1)

    x = embed[tok[:, 0]].double()
    hn = norm(x)
    q = rope(lin("q", hn).view(B, 32, 128))
    kn, vn = rope(lin("k", hn).view(B, 8, 128)), lin("v", hn).view(B, 8, 128)
    kc, vc = k.double(), v.double()
    kc[:, :, pos], vc[:, :, pos] = kn, vn
    a = torch.stack([_attend(q[i].unsqueeze(1), kc[i], vc[i], 128 ** -0.5, pos)[:, 0] for i in range(B)])
    x = x + lin("o", a.reshape(B, 4096))
    hn = norm(x)
    x = x + lin("down", F.silu(lin("gate", hn)) * lin("up", hn))
    return [lin("head", norm(x)), kn, vn]


def exact(case, seed):
    kind = case["kind"]
    if kind == "llama":
        return _exact_llama(case, seed)
    ins = _inputs(case, seed)
    if kind == "linear":
        x, w, bias = ins
        w = w.double()
        y = x.double() @ (w.t().contiguous() if case["layout"] == "nk" else w)
        return y if bias is None else y + bias.double()
    if kind == "qlinear":
        x, w, s, b = ins
        return x.double() @ _dequant(w, s, b, case["bits"], case["gs"]).t().contiguous()
    if kind == "bmm":
        a, b = ins
        b = b.double()
        return torch.matmul(a.double(), b.transpose(1, 2).contiguous() if case["trans"] else b)
    if kind in ("decode", "prefill"):
        q, k, v, table = ins
        B, Tq = case["B"], case.get("Tq", 1)
        lens = _lens(case, seed).tolist() if kind == "decode" or case["ragged"] else [case["L"]] * B
        out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
        for i in range(B):
            n = lens[i]
            if table is None:
                ki, vi = k[i, :, :n], v[i, :, :n]
            else:
                pages = table[i].long()
                ki = k[pages].transpose(0, 1).reshape(case["Hkv"], -1, case["D"])[:, :n]
                vi = v[pages].transpose(0, 1).reshape(case["Hkv"], -1, case["D"])[:, :n]
            out[i] = _attend(q[i].double(), ki.double(), vi.double(), case["D"] ** -0.5, n - Tq)
        return out
    x, w, b = (t.double() for t in ins)
    rms = x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w
    c = x - x.mean(-1, keepdim=True)
    return [rms, c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5) * w + b]
