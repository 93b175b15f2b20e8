"""What the fused RoPE and K/V cache write refuses, on the host: nothing is
launched (validation comes before the library is called)."""

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


def test_caches_an_assignment_refuses():
    """A cache broadcast over its batch, and an inference tensor outside
    inference mode, are left to the slice assignment, which raises."""
    from mlx_batch_invariant_amd.llama import _writable
    c = torch.zeros(1, 2, 8, 32)
    assert _writable(c) and _writable(c.transpose(1, 2)) and _writable(c[:, :, 2:])
    assert _writable(c[:, :1].expand(1, 1, 8, 32))
    assert not _writable(c.expand(3, 2, 8, 32)) and not _writable(c[:, :1].expand(1, 4, 8, 32))
    with torch.inference_mode():
        i = torch.zeros(1, 2, 8, 32)
        assert _writable(i)
    assert not _writable(i)
    for bad in (c.expand(3, 2, 8, 32), i):
        with pytest.raises(RuntimeError):
            bad[:, :, 1:2] = torch.ones(bad.shape[0], 2, 1, 32)
