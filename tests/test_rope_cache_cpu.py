"""What the fused RoPE and K/V cache write refuses, on the host: nothing is
launched (validation comes before the library is called)."""

import numpy as np
import pytest
import torch


def _operands(B=2, T=3, Hq=4, Hkv=2, D=32, L=8):
    q, k, v = (torch.zeros(B, T, h, D) for h in (Hq, Hkv, Hkv))
    return q, k, v, torch.zeros(B, Hkv, L, D), torch.zeros(B, Hkv, L, D)


@pytest.mark.parametrize("shape", [(2, 1, 3, 16), (1, 16), (16,), (3, 32), (4, 16), (1, 3, 16)])
def test_tables_of_another_shape_are_refused(shape):
    """The kernel reads [T, D / 2] from the pointers whatever the tensors are:
    tables that broadcast (a row per sequence, one row for all tokens) or are
    of another size never reach it."""
    from mlx_batch_invariant_amd.llama import _tables_fit, rope_cache
    q, k, v, kc, vc = _operands()
    good, bad = torch.zeros(3, 16), torch.zeros(shape)
    assert _tables_fit(q, good, good)
    for cos, sin in ((bad, bad), (good, bad), (bad, good)):
        assert not _tables_fit(q, cos, sin)
        with pytest.raises(ValueError, match="tables"):
            rope_cache(q, k, v, cos, sin, kc, vc, 0)


@pytest.mark.parametrize("pos", [6, np.int64(6), torch.tensor(6)])
def test_position_of_any_integer_type(pos, monkeypatch):
    """Every integer a slice takes reaches the library's own check (rows past
    the cache here) instead of failing in the argument conversion."""
    from mlx_batch_invariant_amd import _lib
    from mlx_batch_invariant_amd.llama import rope_cache
    monkeypatch.setattr(_lib, "stream_of", lambda t: None)      # host tensors have no stream
    q, k, v, kc, vc = _operands()
    with pytest.raises(ValueError, match="pos=6 max_len=8"):
        rope_cache(q, k, v, torch.zeros(3, 16), torch.zeros(3, 16), kc, vc, pos)
