"""The dense tiles that take a batch of matrices in one grid, a row-major
right-hand side and a K that is not a multiple of 64: bit for bit the one-row
launches on a contiguous transposed copy (which the oracle tests pin), at the
edges of each tile form, and over the strides the entry points accept."""

import pytest
import torch

from helpers import DT, bits, gen, randn

pytestmark = pytest.mark.gpu


def _bi():
    import mlx_batch_invariant_amd as bi
    return bi


def _one_row(a, bt, r):
    """Row r of a @ bt.T by the M = 1 launch on padded contiguous operands."""
    K = a.shape[1]
    K8 = (K + 7) // 8 * 8
    ap = torch.zeros((1, K8), dtype=a.dtype, device=a.device)
    bp = torch.zeros((bt.shape[0], K8), dtype=a.dtype, device=a.device)
    ap[:, :K], bp[:, :K] = a[r:r + 1], bt
    return _bi().batch_invariant_matmul(ap, bp.t())


def _check_rows(out, a, bt, rows):
    for r in sorted(set(rows)):
        assert bits(out[r:r + 1]) == bits(_one_row(a, bt, r)), f"row {r}"


# (M, N, K): every tile form's edges, K tails of 8 .. 56 past a stage and short
# of a group, fewer columns than a tile, split K (few tiles).
_SHAPES = [(1, 8, 8), (1, 1024, 4096), (31, 64, 72), (33, 96, 264), (64, 200, 1000), (65, 72, 520), (128, 1024, 776),
           (129, 4096, 1032), (515, 4096, 1064), (300, 14336, 136), (2049, 3080, 1048), (700, 40, 2088)]


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", _SHAPES)
def test_row_major_rhs_equals_transposed(dt, M, N, K):
    g = gen(M + N + K)
    a = randn((M, K), DT[dt], g)
    b = randn((K, N), DT[dt], g, 0.1)
    got = _bi().batch_invariant_matmul(a, b)
    _check_rows(got, a, b.t(), [0, M // 2, M - 1, min(M - 1, 63), min(M - 1, 128)])


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [s for s in _SHAPES if s[0] > 32])
def test_ragged_k_equals_one_row(dt, M, N, K):
    g = gen(M + 2 * N + K)
    a = randn((M, K), DT[dt], g)
    bt = randn((N, K), DT[dt], g, 0.1)
    got = _bi().batch_invariant_matmul(a, bt.t())
    _check_rows(got, a, bt, [0, M // 2, M - 1, min(M - 1, 63), min(M - 1, 128)])


def test_row_major_views_and_padding():
    """Offsets, row gaps (which hold NaN), odd K and odd N, non-finite values
    next to the operands: only the operands' own elements count."""
    g = gen(5)
    for M, N, K in [(40, 100, 72), (3, 64, 65), (130, 77, 200), (70, 136, 133)]:
        a = randn((M, K), torch.bfloat16, g)
        b = randn((K, N), torch.bfloat16, g)
        abig = torch.full((M + 2, K + 40), float("nan"), dtype=torch.bfloat16, device="cuda")
        bbig = torch.full((K + 3, (N + 7) // 8 * 8 + 24), float("nan"), dtype=torch.bfloat16, device="cuda")
        av, bv = abig[1:M + 1, 8:K + 8], bbig[1:K + 1, 16:N + 16]
        av.copy_(a)
        bv.copy_(b)
        want = _bi().batch_invariant_matmul(a, b.t().contiguous().t())
        for x in (a, av):
            for y in (b, bv):
                assert bits(_bi().batch_invariant_matmul(x, y)) == bits(want), (M, N, K)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("row_major", [False, True])
@pytest.mark.parametrize("batch,M,N,K", [(2, 1, 64, 8), (5, 17, 96, 264), (3, 64, 72, 520), (48, 33, 64, 136),
                                         (7, 200, 72, 1032), (70, 128, 128, 64), (130, 300, 40, 72), (9, 520, 520, 200)])
def test_batched_equals_slices(dt, row_major, batch, M, N, K):
    g = gen(batch + M + N + K)
    a = randn((batch, M, K), DT[dt], g)
    b = randn((batch, K, N) if row_major else (batch, N, K), DT[dt], g, 0.1)
    got = _bi().batch_invariant_bmm(a, b if row_major else b.transpose(1, 2))
    for i in sorted({0, 1, batch // 2, batch - 1}):
        bt = (b[i].t() if row_major else b[i])
        _check_rows(got[i], a[i], bt, [0, M // 2, M - 1])


def test_batched_broadcast_and_sliced_operands():
    """Zero batch strides, head-sliced views and an odd inner size through
    torch.matmul's batch rules."""
    g = gen(11)
    a = randn((2, 6, 50, 72), torch.float16, g)
    kv = randn((2, 90, 6, 3, 72), torch.float16, g)          # [B, L, H, parts, D]
    k, v = kv[:, :, :, 0].permute(0, 2, 3, 1), kv[:, :, :, 1].permute(0, 2, 1, 3)
    s = _bi().batch_invariant_bmm(a, k)                       # [2, 6, 50, 90]
    o = _bi().batch_invariant_bmm(s[..., :89], v[..., :89, :])
    w = randn((72, 40), torch.float16, g)
    c = _bi().batch_invariant_bmm(a, w)
    for i, h in [(0, 0), (1, 5)]:
        assert bits(s[i, h]) == bits(_bi().batch_invariant_matmul(a[i, h], k[i, h]))
        _check_rows(s[i, h], a[i, h], k[i, h].t(), [0, 49])
        _check_rows(o[i, h], s[i, h, :, :89], v[i, h, :89].t(), [0, 49])
        _check_rows(c[i, h], a[i, h], w.t(), [0, 49])


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("shape,cut", [((1, 1), (0, 0)), ((3, 7), (0, 0)), ((5, 9), (1, 3)), ((130, 65), (2, 1)),
                                       ((2, 33, 100), (1, 5)), ((70, 3, 31), (0, 2))])
def test_pad_rows_copies_exactly(dt, shape, cut):
    """Every row length and alignment, views with gaps and offsets (the gaps
    hold NaN), a broadcast batch: the rows, then zeros."""
    from mlx_batch_invariant_amd.kernels.matmul import _pad_rows
    big = torch.full((*shape[:-1], shape[-1] + 11), float("nan"), dtype=DT[dt], device="cuda")
    t = big[..., cut[1]:cut[1] + shape[-1]][..., cut[0]:, :]
    t.copy_(randn(tuple(t.shape), DT[dt], gen(shape[-1])))
    for C in ((shape[-1] + 7) // 8 * 8, (shape[-1] + 7) // 8 * 8 + 16):
        want = torch.zeros((*t.shape[:-1], C), dtype=DT[dt], device="cuda")
        want[..., :shape[-1]] = t
        assert bits(_pad_rows(t, C)) == bits(want)
    if t.ndim == 2:
        assert bits(_pad_rows(t.expand(4, *t.shape), C)) == bits(want.expand(4, *want.shape))


@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_rows_far_apart_row_major(dt):
    """Rows 2^22 elements apart: one row in place (the last token of a prompt,
    x[:, -1]), several rows through a copy, 2-D and batched."""
    g = gen(11)
    h = torch.zeros((2, 1024, 4096), dtype=DT[dt], device="cuda")
    h[:, -1] = randn((2, 4096), DT[dt], g)
    w = randn((4096, 72), DT[dt], g, 0.1)
    want = _bi().batch_invariant_matmul(h[:, -1].contiguous(), w)
    for x in (h[:1, -1], h[:, -1], h[:, -1][:, :4096]):
        assert x.stride(0) == 1 << 22
        assert bits(_bi().batch_invariant_matmul(x, w)) == bits(want[:x.shape[0]])
        b3 = w.expand(1, -1, -1)
        assert bits(_bi().batch_invariant_bmm(x[None], b3)[0]) == bits(want[:x.shape[0]])
    b3 = w.expand(2, -1, -1).contiguous()
    assert bits(_bi().batch_invariant_bmm(h[:, -1:], b3)) == bits(want[:, None])


def test_odd_columns_row_major():
    """b [K, N] with an odd N or an unaligned base takes a row-padded copy."""
    g = gen(2)
    for M, N, K in [(1, 33, 100), (70, 1001, 264), (300, 65, 72)]:
        a, b = randn((M, K), torch.float16, g), randn((K, N + 3), torch.float16, g)
        for y in (b[:, :N], b[:, 3:]):
            got = _bi().batch_invariant_matmul(a, y)
            _check_rows(got, a, y.t(), [0, M - 1])
        a3, b3 = randn((3, M, K), torch.float16, g), randn((3, K, N), torch.float16, g)
        got = _bi().batch_invariant_bmm(a3, b3)
        _check_rows(got[2], a3[2], b3[2].t(), [0, M - 1])


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("M,N,K", [(1, 1, 8), (1, 33, 264), (17, 64, 256), (33, 130, 520), (300, 65, 72)])
def test_direct_call_equals_general(dt, M, N, K):
    """x @ W.T passed on at once, and the same product through the general path:
    whole operands, aligned row slices with gaps, and what is not taken at once
    (an odd base, row strides of 4 mod 8, a row stride below K, mixed types)."""
    from mlx_batch_invariant_amd.kernels.matmul import _matmul_direct, matmul_bt
    g = gen(4)
    a0, w0 = randn((M, K), DT[dt], g), randn((N, K), DT[dt], g)
    x, w = randn((M + 1, K + 20), DT[dt], g), randn((N + 1, K + 20), DT[dt], g)
    want = matmul_bt(a0, w0)
    assert bits(_matmul_direct(a0, w0.t())) == bits(want)
    x8, w8 = randn((M + 1, K + 24), DT[dt], g), randn((N + 1, K + 24), DT[dt], g)
    a, wv = x8[1:, 8:8 + K], w8[1:, 16:16 + K]
    a.copy_(a0)
    wv.copy_(w0)
    assert bits(_matmul_direct(a, wv.t())) == bits(want)
    assert bits(_bi().batch_invariant_matmul(a, wv.t())) == bits(want)
    for y, v in [(x[1:, 1:1 + K], w0), (a0, w[1:, 4:4 + K]), (x[1:, 4:4 + K], w[1:, 4:4 + K])]:
        assert _matmul_direct(y, v.t()) is None
        want4 = matmul_bt(y.contiguous(), v.contiguous())
        assert bits(_bi().batch_invariant_matmul(y, v.t())) == bits(want4)
        y3, v3 = y.expand(2, -1, -1), v.t().expand(2, -1, -1)
        assert bits(_bi().batch_invariant_bmm(y3, v3)) == bits(want4.expand(2, -1, -1))
    assert _matmul_direct(a0[:1].expand(2, K), w0.t()) is None
    assert _matmul_direct(a0, w0.t().double()) is None and _matmul_direct(a0.cpu(), w0.cpu().t()) is None
    assert bits(_bi().batch_invariant_matmul(a0[:1].expand(2, K), w0.t())[1]) == bits(matmul_bt(a0[:1], w0)[0])


def test_direct_call_with_repacked_weights(monkeypatch):
    """The direct call looks a weight's repacked copy up itself, and a copy kept
    for one weight leaves the others' calls as they were; a stale copy is not
    used. Same bits each way."""
    from mlx_batch_invariant_amd import _lib
    from mlx_batch_invariant_amd.kernels import matmul as km
    bi = _bi()
    g = gen(5)
    w, other = randn((72, 512), torch.bfloat16, g), randn((72, 512), torch.bfloat16, g)
    x = randn((17, 512), torch.bfloat16, g)
    want, want_other = bi.batch_invariant_matmul(x, w.t()), bi.batch_invariant_matmul(x, other.t())
    packed = []
    real = _lib.load().bi_matmul_packed
    monkeypatch.setattr(_lib.load(), "bi_matmul_packed", lambda *a: packed.append(a[6]) or real(*a))
    bi.cache_packed_weight(w)
    try:
        for M in (1, 16, 17):
            assert bits(km._matmul_direct(x[:M], w.t())) == bits(want[:M])
            assert bits(km._matmul_direct(x[:M], other.t())) == bits(want_other[:M])
        assert packed == [1, 16]
        assert bits(km._matmul_direct(x[:4], w[:40].t())) == bits(want[:4, :40])     # another weight's shape
        w.mul_(2)
        assert bits(km._matmul_direct(x[:4], w.t())) == bits(bi.batch_invariant_matmul(x, w.t())[:4])
        assert packed == [1, 16]
    finally:
        bi.drop_packed_weight(w)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("B,M,N,K", [(2, 1, 64, 1032), (31, 16, 64, 1024), (32, 16, 64, 1024), (3, 33, 130, 4100),
                                     (64, 64, 8, 776), (65, 64, 64, 776), (2, 65, 130, 20000), (4, 200, 72, 1280),
                                     (17, 129, 64, 1000), (2, 300, 96, 520)])
def test_small_batches_with_long_k(dt, B, M, N, K):
    """Row-major batches that split K and their neighbours that do not: the
    lines of the rule, partial groups, several K chunks per slice, a broadcast
    operand."""
    g = gen(B + M + K)
    a = randn((B, M, K), DT[dt], g)
    b = randn((B, K, N), DT[dt], g, 0.1)
    got = _bi().batch_invariant_bmm(a, b)
    one = _bi().batch_invariant_bmm(a, b[:1].expand(B, K, N))
    for i in {0, B // 2, B - 1}:
        _check_rows(got[i], a[i], b[i].t(), [0, M // 2, M - 1])
        _check_rows(one[i], a[i], b[0].t(), [M - 1])


@pytest.mark.parametrize("M", [1, 40, 200])
def test_small_batch_without_workspace(M):
    """A batch that splits K runs unsplit, with the same bits, where the caller
    brings no workspace, a short one or a misaligned one."""
    bi = _bi()
    lib = bi._lib.load()
    g = gen(M)
    B, N, K = 2, 72, 2048
    a, b = randn((B, M, K), torch.bfloat16, g), randn((B, K, N), torch.bfloat16, g, 0.1)
    want = bi.batch_invariant_bmm(a, b)
    need = lib.bi_matmul_kn_workspace_bytes(B, M, N, K)
    assert need > 0
    ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
    for ptr, n in ((None, 0), (ws.data_ptr(), need - 16), (ws.data_ptr() + 8, need), (ws.data_ptr(), need)):
        out = torch.empty_like(want)
        bi._lib.check(lib.bi_matmul_kn(a.data_ptr(), M * K, K, b.data_ptr(), K * N, N, out.data_ptr(), M * N, B, M, N, K,
                                       bi._lib.BI_BF16, ptr, n, bi._lib.stream_of(a)), "bi_matmul_kn")
        assert bits(out) == bits(want)


def test_pad_rows_past_one_launch():
    """More 16-byte pieces than one launch has threads (2^32): 64 GiB of output
    from one broadcast row, the rows at both ends of every launch."""
    from mlx_batch_invariant_amd.kernels.matmul import _pad_rows
    free = torch.cuda.mem_get_info()[0]
    if free < 90 << 30:
        pytest.skip(f"{free >> 30} GiB of GPU memory free, 90 needed")
    R, step = (1 << 32) // 3 + 1000, (1 << 31) // 3
    row = torch.arange(1, 18, dtype=torch.bfloat16, device="cuda")
    out = _pad_rows(row.expand(R, 17), 24)
    want = torch.zeros(24, dtype=torch.bfloat16, device="cuda")
    want[:17] = row
    for r in (0, 1, step - 1, step, 2 * step - 1, 2 * step, R - 1):
        assert bits(out[r]) == bits(want), r
    assert bool((out[::4099] == want).all())
    del out
    torch.cuda.empty_cache()
