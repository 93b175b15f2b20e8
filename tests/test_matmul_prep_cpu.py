"""How the matmul wrappers prepare their operands, on the host."""

import pytest
import torch


@pytest.mark.parametrize("M,stride", [(1, 1 << 22), (1, 64), (1, 5_000_000), (3, 1 << 22), (3, 72)])
def test_row_stride_passed_to_the_row_major_product(M, stride):
    """The stride bi_matmul_kn is given stays below its limit for any view, a
    single row included (its stride counts as contiguous whatever it is)."""
    from mlx_batch_invariant_amd.kernels.matmul import _MAX_LD, _rows_within
    x = torch.arange(1, 1 + M * stride, dtype=torch.int16).view(1, M, stride)[:, :, :64]
    y, ld = _rows_within(x, 64)
    assert 64 <= ld < _MAX_LD and ld % 8 == 0
    assert torch.equal(y, x) and (M == 1 or y.stride(1) == ld)
    assert (y.data_ptr() == x.data_ptr()) == (M == 1 or stride < _MAX_LD)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_rows_taken_in_place_are_what_the_library_takes(dt):
    """Row strides of 4 mod 8 elements are 16-byte aligned in fp32, but the
    library takes multiples of 8 only."""
    from mlx_batch_invariant_amd.kernels.matmul import _kcontig, _prep_batched
    for ld, ok in ((28, False), (32, True)):
        x = torch.zeros((3, ld), dtype=dt)[1:, 8:16]
        assert _kcontig(x) is ok
        if ok:
            assert _prep_batched(x[None], 8).data_ptr() == x.data_ptr()
