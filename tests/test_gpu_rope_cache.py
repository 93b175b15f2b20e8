"""RoPE and the K/V cache writes in one launch against the elementwise ops, bit
for bit, over types, head sizes, token counts and cache layouts."""

import numpy as np
import pytest
import torch

from helpers import DT, bits, gen, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("B,T,Hq,Hkv,D,pos", [(1, 1, 32, 8, 128, 0), (3, 5, 4, 2, 64, 11), (2, 37, 3, 1, 16, 3),
                                              (5, 1, 14, 2, 96, 62)])
@pytest.mark.parametrize("token_major", [False, True])
def test_rope_cache_equals_elementwise(dt, B, T, Hq, Hkv, D, pos, token_major):
    from mlx_batch_invariant_amd import set_batch_invariant_mode
    from mlx_batch_invariant_amd.llama import _fused_rope_ok, _rope, rope_cache
    g = gen(B + T + D)
    q, k, v = (randn((B, T, h, D), DT[dt], g, 3.0) for h in (Hq, Hkv, Hkv))
    ang = torch.rand((T, D // 2), generator=g) * 6.3
    cos, sin = ang.cos().to(DT[dt]).cuda(), ang.sin().to(DT[dt]).cuda()
    L = pos + T + 2
    shape = (B + 1, L, Hkv, D) if token_major else (B + 1, Hkv, L, D)
    base = [randn(shape, DT[dt], g) for _ in range(2)]
    view = lambda c: (c.permute(0, 2, 1, 3) if token_major else c)[1:]       # a slice of a larger cache
    want = [c.clone() for c in base]
    qw = _rope(q.transpose(1, 2), cos, sin)
    view(want[0])[:, :, pos:pos + T] = _rope(k.transpose(1, 2), cos, sin)
    view(want[1])[:, :, pos:pos + T] = v.transpose(1, 2)
    assert not _fused_rope_ok(q, k, v, cos, sin, view(base[0]), view(base[1]), pos)      # outside the mode
    with set_batch_invariant_mode():
        assert _fused_rope_ok(q, k, v, cos, sin, view(base[0]), view(base[1]), pos)
        assert not _fused_rope_ok(q, k, v, cos, sin, view(base[0]), view(base[1]), L)    # past the cache
        assert not _fused_rope_ok(q.transpose(1, 2).contiguous().transpose(1, 2), k, v, cos, sin, view(base[0]),
                                  view(base[1]), pos) or T == 1
    got = rope_cache(q, k, v, cos, sin, view(base[0]), view(base[1]), pos)
    assert bits(got) == bits(qw)
    for a, b in zip(base, want):
        assert bits(a) == bits(b)                                            # every other row untouched


@pytest.mark.parametrize("pos", [3, np.int64(3), torch.tensor(3), -6])
def test_block_position_forms(pos):
    """Positions of any integer type, and rows counted from the cache's end."""
    from mlx_batch_invariant_amd import set_batch_invariant_mode
    from mlx_batch_invariant_amd.llama import Block, LlamaConfig
    cfg = LlamaConfig(vocab=64, hidden=128, ffn=256, layers=1, heads=2, kv_heads=1, head_dim=64, bits=None)
    g = gen(9)
    blk = Block(cfg, torch.Generator(device="cuda").manual_seed(0), "cuda", torch.bfloat16)
    x = randn((2, 1, cfg.hidden), torch.bfloat16, g)
    cos, sin = randn((1, 32), torch.bfloat16, g), randn((1, 32), torch.bfloat16, g)
    base = [randn((2, 1, 9, 64), torch.bfloat16, g) for _ in range(2)]

    def run(pos):
        cache = [c.clone() for c in base]
        with torch.no_grad(), set_batch_invariant_mode():
            return [blk(x, cos, sin, cache, pos), *cache]

    for a, b in zip(run(pos), run(3)):                 # row -6 of 9 is row 3
        assert bits(a) == bits(b)


def test_rope_cache_counts_as_an_in_place_change():
    """The caches' version counters move, so a graph that saved a cache for its
    backward pass notices the write; caches made in inference mode have none."""
    from mlx_batch_invariant_amd.llama import rope_cache
    g = gen(10)
    q, k, v = (randn((1, 2, h, 64), torch.bfloat16, g) for h in (4, 2, 2))
    cs = randn((2, 32), torch.bfloat16, g)
    kc, vc = (torch.zeros(1, 2, 6, 64, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    w = torch.ones_like(kc, requires_grad=True)
    y = (w * kc).sum()
    before = kc._version, vc._version
    rope_cache(q, k, v, cs, cs, kc, vc, 1)
    assert kc._version > before[0] and vc._version > before[1]
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward()
    with torch.inference_mode():
        ki, vi = torch.zeros_like(kc), torch.zeros_like(vc)
        rope_cache(q, k, v, cs, cs, ki, vi, 1)
    assert bits(ki) == bits(kc) and bits(vi) == bits(vc)


def test_block_refuses_caches_an_assignment_refuses():
    from mlx_batch_invariant_amd import set_batch_invariant_mode
    from mlx_batch_invariant_amd.llama import Block, LlamaConfig
    cfg = LlamaConfig(vocab=64, hidden=128, ffn=256, layers=1, heads=2, kv_heads=1, head_dim=64, bits=None)
    blk = Block(cfg, torch.Generator(device="cuda").manual_seed(0), "cuda", torch.bfloat16)
    x = torch.zeros((2, 1, cfg.hidden), dtype=torch.bfloat16, device="cuda")
    cs = torch.zeros((1, 32), dtype=torch.bfloat16, device="cuda")
    new = lambda n: torch.zeros((n, 1, 4, 64), dtype=torch.bfloat16, device="cuda")
    with torch.inference_mode():
        inference = new(2)
    for bad in (new(1).expand(2, 1, 4, 64), inference):
        for cache in ((bad, new(2)), (new(2), bad)):
            with torch.no_grad(), set_batch_invariant_mode(), pytest.raises(RuntimeError):
                blk(x, cs, cs, cache, 1)


def test_rope_cache_rejects():
    from mlx_batch_invariant_amd.llama import rope_cache
    q, k = torch.zeros(1, 2, 4, 64, device="cuda"), torch.zeros(1, 2, 2, 64, device="cuda")
    cs, c = torch.zeros(2, 32, device="cuda"), torch.zeros(1, 2, 3, 64, device="cuda")
    with pytest.raises(ValueError, match="bad shape"):
        rope_cache(q, k, k, cs, cs, c, c.clone(), 2)                         # rows past the cache


def test_block_tables_of_another_shape_broadcast():
    """Tables with a position per sequence ([B, 1, T, D / 2]) and with one row
    for every token ([1, D / 2]) broadcast as in the elementwise ops: each
    sequence gets what it gets alone with its own [T, D / 2] tables."""
    from mlx_batch_invariant_amd import set_batch_invariant_mode
    from mlx_batch_invariant_amd.llama import Block, LlamaConfig
    cfg = LlamaConfig(vocab=64, hidden=256, ffn=512, layers=1, heads=4, kv_heads=2, head_dim=64, bits=None)
    B, T, L = 3, 5, 9
    g = gen(8)
    blk = Block(cfg, torch.Generator(device="cuda").manual_seed(0), "cuda", torch.bfloat16)
    x = randn((B, T, cfg.hidden), torch.bfloat16, g)
    ang = torch.rand((B, 1, T, cfg.head_dim // 2), generator=g) * 6.3
    ang1 = ang[0, 0, :1]

    def run(x, ang):
        cache = [torch.zeros(x.shape[0], cfg.kv_heads, L, cfg.head_dim, dtype=x.dtype, device="cuda") for _ in range(2)]
        cos, sin = (f(ang).to(torch.bfloat16).cuda() for f in (torch.cos, torch.sin))
        with torch.no_grad(), set_batch_invariant_mode():
            return [blk(x, cos, sin, cache, 0), *cache]

    got = run(x, ang)
    for b in range(B):
        for u, w in zip(got, run(x[b:b + 1], ang[b, 0])):
            assert bits(u[b:b + 1]) == bits(w)
    for u, w in zip(run(x, ang1), run(x, ang1.expand(T, -1))):
        assert bits(u) == bits(w)
