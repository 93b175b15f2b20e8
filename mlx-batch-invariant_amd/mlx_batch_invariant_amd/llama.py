"""A random-initialised Llama-3-8B-shaped decoder built from stock torch
modules, used to check that the four batch-invariant ops compose.

Every matmul goes through ``nn.Linear`` / ``F.linear`` (or this package's
``QuantizedLinear`` for MLX-affine weights), every norm through ``nn.RMSNorm``
and attention through ``F.scaled_dot_product_attention``, so the model is the
stock path outside ``set_batch_invariant_mode`` and the batch-invariant kernels
inside it, with no code change: the drop-in property the reference checks
end to end with ``harness/model_sweep.py`` (row-0 logits / per-block hashes at
batch 1, 4, 16, 64, prefill and cached decode; :62-108).

Prefill is causal over the prompt (``is_causal``; a later chunk of a chunked
prefill uses ``causal_lower_right``); decode steps attend to a preallocated KV
cache through a view (no copy), one token per sequence. RoPE (theta 5e5),
SiLU-gated MLP and residual adds are elementwise torch ops, which compute each
element from its own inputs only.
"""

from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.nn.functional as F
from torch.nn.attention.bias import causal_lower_right

from . import _lib, _mode
from .nn import QuantizedLinear


@dataclass
class LlamaConfig:
    vocab: int = 128256
    hidden: int = 4096
    ffn: int = 14336
    layers: int = 32
    heads: int = 32
    kv_heads: int = 8
    head_dim: int = 128
    rope_theta: float = 5e5
    eps: float = 1e-5
    bits: int | None = 4          # None: bf16 linears
    group_size: int = 64


def _linear(cfg: LlamaConfig, fin: int, fout: int, gen: torch.Generator, device, dtype):
    """``nn.Linear`` (bf16 run) or ``QuantizedLinear`` quantized from it, with
    N(0, 0.02^2) weights drawn on ``device``."""
    lin = torch.nn.Linear(fin, fout, bias=False, device="meta", dtype=dtype)
    w = (torch.randn((fout, fin), generator=gen, device=device) * 0.02).to(dtype)
    lin.weight = torch.nn.Parameter(w, requires_grad=False)
    if cfg.bits is None:
        return lin
    q = QuantizedLinear.from_linear(lin, group_size=cfg.group_size, bits=cfg.bits)
    del lin, w
    return q


class Block(torch.nn.Module):
    def __init__(self, cfg: LlamaConfig, gen, device, dtype):
        super().__init__()
        h, kvd = cfg.hidden, cfg.kv_heads * cfg.head_dim
        self.cfg = cfg
        self.attn_norm = torch.nn.RMSNorm(h, eps=cfg.eps, device=device, dtype=dtype)
        self.mlp_norm = torch.nn.RMSNorm(h, eps=cfg.eps, device=device, dtype=dtype)
        self.q = _linear(cfg, h, cfg.heads * cfg.head_dim, gen, device, dtype)
        self.k = _linear(cfg, h, kvd, gen, device, dtype)
        self.v = _linear(cfg, h, kvd, gen, device, dtype)
        self.o = _linear(cfg, cfg.heads * cfg.head_dim, h, gen, device, dtype)
        self.gate = _linear(cfg, h, cfg.ffn, gen, device, dtype)
        self.up = _linear(cfg, h, cfg.ffn, gen, device, dtype)
        self.down = _linear(cfg, cfg.ffn, h, gen, device, dtype)

    def forward(self, x, cos, sin, cache, pos):
        cfg = self.cfg
        B, T, _ = x.shape
        hn = self.attn_norm(x)
        q = self.q(hn).view(B, T, cfg.heads, cfg.head_dim)
        k = self.k(hn).view(B, T, cfg.kv_heads, cfg.head_dim)
        v = self.v(hn).view(B, T, cfg.kv_heads, cfg.head_dim)
        kc, vc = cache
        if _fused_rope_ok(q, k, v, cos, sin, kc, vc, pos):
            q = rope_cache(q, k, v, cos, sin, kc, vc, pos)
        else:
            q = _rope(q.transpose(1, 2), cos, sin)
            kc[:, :, pos:pos + T] = _rope(k.transpose(1, 2), cos, sin)
            vc[:, :, pos:pos + T] = v.transpose(1, 2)
        L = pos + T
        if T == 1:
            mask = {}
        elif pos == 0:
            mask = {"is_causal": True}
        else:                                   # chunked prefill: chunk t sees keys <= pos + t
            mask = {"attn_mask": causal_lower_right(T, L)}
        a = F.scaled_dot_product_attention(q, kc[:, :, :L], vc[:, :, :L], enable_gqa=True, **mask)
        x = x + self.o(a.transpose(1, 2).reshape(B, T, cfg.heads * cfg.head_dim))
        hn = self.mlp_norm(x)
        x = x + self.down(F.silu(self.gate(hn)) * self.up(hn))
        return x


def _rope(x, cos, sin):
    x1, x2 = x[..., : x.shape[-1] // 2], x[..., x.shape[-1] // 2:]
    return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], dim=-1)


def _fused_rope_ok(q, k, v, cos, sin, kc, vc, pos) -> bool:
    """Whether ``rope_cache`` takes a block's tensors (under the mode, on the
    GPU, one dtype, 16-byte aligned rows, one table row per token, no gradient
    to record). Tables that broadcast (one position per sequence, one row for
    every token) take the elementwise ops."""
    ts = (q, k, v, cos, sin, kc, vc)
    dt, D = q.dtype, q.shape[-1]
    if not _tables_fit(q, cos, sin):
        return False
    unit = 16 // q.element_size() if dt in _lib.FLOAT_DTYPES else 0
    if not unit or not _mode.is_batch_invariant_mode_enabled() or D % 16:
        return False
    if pos < 0 or pos + q.shape[1] > min(kc.shape[2], vc.shape[2]):     # a slice counts rows below 0 from the end
        return False
    if torch.is_grad_enabled() and any(t.requires_grad for t in ts):
        return False
    if any(type(t) is not torch.Tensor or not t.is_cuda or t.dtype != dt or t.device != q.device or t.data_ptr() % 16
           for t in ts):
        return False
    if not all(_writable(c) for c in (kc, vc)):
        return False
    if q.numel() + 2 * k.numel() > 16 * ((1 << 32) - 256):               # elements of one launch
        return False
    # rows [b, t] at one stride with contiguous heads; contiguous tables; caches with contiguous d
    rows = all(t.is_contiguous() for t in (q, k, v, cos, sin))
    return rows and all(c.stride(3) == 1 and all(s % unit == 0 for s in c.stride()[:3])
                        and c.shape[0] == q.shape[0] and c.shape[1] == k.shape[2] and c.shape[3] == D for c in (kc, vc))


def _tables_fit(q, cos, sin) -> bool:
    """cos and sin are [T, D / 2] for q [B, T, heads, D]: row t of the tables is
    token t's, in every sequence (the kernel sees pointers only)."""
    return tuple(cos.shape) == tuple(sin.shape) == (q.shape[1], q.shape[3] // 2)


def _writable(c) -> bool:
    """No stride-0 dimension (rows that share memory) and no inference tensor
    outside inference mode: what a slice assignment into ``c`` refuses."""
    return (all(s > 0 or n <= 1 for s, n in zip(c.stride(), c.shape))
            and (not c.is_inference() or torch.is_inference_mode_enabled()))


def rope_cache(q, k, v, cos, sin, kc, vc, pos):
    """One launch (``bi_rope_cache``) for ``_rope`` of q and k and the writes of
    the rotated keys and the values into rows ``pos ..`` of the caches: the bits
    of those elementwise ops. Returns q rotated, ``[B, heads, T, D]``. The
    caches count as changed in place (their version counters), as by the writes."""
    B, T, Hq, D = q.shape
    Hkv = k.shape[2]
    if not _tables_fit(q, cos, sin):
        raise ValueError(f"rope_cache: tables {tuple(cos.shape)} and {tuple(sin.shape)}; need ({T}, {D // 2}) each")
    out = torch.empty((B, Hq, T, D), dtype=q.dtype, device=q.device)
    strides = (_lib._c_i64 * 6)(*kc.stride()[:3], *vc.stride()[:3])
    rc = _lib.load().bi_rope_cache(q.data_ptr(), Hq * D, k.data_ptr(), Hkv * D, v.data_ptr(), Hkv * D, cos.data_ptr(),
                                   sin.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), B, T, Hq, Hkv, D, pos,
                                   min(kc.shape[2], vc.shape[2]), strides, _lib.DTYPE_CODE[q.dtype], _lib.stream_of(q))
    _lib.check(rc, "bi_rope_cache")
    torch.autograd.graph.increment_version([c for c in (kc, vc) if not c.is_inference()])
    return out


class LlamaShaped(torch.nn.Module):
    """Decoder with Llama-3-8B shapes (or fewer layers for tests)."""

    def __init__(self, cfg: LlamaConfig, device="cuda", dtype=torch.bfloat16, seed: int = 0):
        super().__init__()
        gen = torch.Generator(device=device).manual_seed(seed)
        self.cfg = cfg
        self.dtype = dtype
        self.embed = (torch.randn((cfg.vocab, cfg.hidden), generator=gen, device=device) * 0.02).to(dtype)
        self.blocks = torch.nn.ModuleList([Block(cfg, gen, device, dtype) for _ in range(cfg.layers)])
        self.norm = torch.nn.RMSNorm(cfg.hidden, eps=cfg.eps, device=device, dtype=dtype)
        self.head = _linear(cfg, cfg.hidden, cfg.vocab, gen, device, dtype)
        self.device = torch.device(device)

    def _ensure_rope(self, n: int):
        """cos / sin tables of positions [0, n) on the device (built once, grown
        on demand outside any graph capture; every position's entries are
        computed from that position alone, so a slice equals a fresh table)."""
        have = getattr(self, "_rope_cos", None)
        if have is not None and have.shape[0] >= n:
            return
        cfg = self.cfg
        n = max(n, 2 * (have.shape[0] if have is not None else 0))
        inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, cfg.head_dim, 2, dtype=torch.float64) / cfg.head_dim))
        ang = torch.outer(torch.arange(0, n, dtype=torch.float64), inv)
        self._rope_cos = ang.cos().to(self.dtype).to(self.device)
        self._rope_sin = ang.sin().to(self.dtype).to(self.device)

    def _rope_tables(self, pos, T):
        self._ensure_rope(pos + T)
        return self._rope_cos[pos:pos + T], self._rope_sin[pos:pos + T]

    def new_cache(self, B: int, max_len: int):
        cfg = self.cfg
        self._ensure_rope(max_len)
        shape = (B, cfg.kv_heads, max_len, cfg.head_dim)
        return [(torch.zeros(shape, dtype=self.dtype, device=self.device),
                 torch.zeros(shape, dtype=self.dtype, device=self.device)) for _ in range(cfg.layers)]

    @torch.no_grad()
    def forward(self, tokens, cache, pos: int, record=None):
        x = self.embed[tokens]
        cos, sin = self._rope_tables(pos, tokens.shape[1])
        for i, blk in enumerate(self.blocks):
            x = blk(x, cos, sin, cache[i], pos)
            if record is not None:
                record.append(x[0:1, -1:].clone())
        return self.head(self.norm(x[:, -1:]))[:, 0]

    @torch.no_grad()
    def generate(self, prompt, steps: int, record=None):
        """Greedy: prefill the prompt, then `steps` cached decode steps.
        Returns (logits of every step [steps+1, B, vocab] for row 0 only, tokens)."""
        B, T = prompt.shape
        cache = self.new_cache(B, T + steps)
        logits = self.forward(prompt, cache, 0, record)
        rows0 = [logits[0:1].clone()]
        tok = logits.argmax(-1, keepdim=True)
        out = [tok]
        for s in range(steps):
            logits = self.forward(tok, cache, T + s, record)
            rows0.append(logits[0:1].clone())
            tok = logits.argmax(-1, keepdim=True)
            out.append(tok)
        return torch.cat(rows0, 0), torch.cat(out, 1)


def param_bytes(model: LlamaShaped) -> int:
    n = 0
    for t in list(model.parameters()) + list(model.buffers()):
        n += t.numel() * t.element_size()
    return n + model.embed.numel() * model.embed.element_size()
