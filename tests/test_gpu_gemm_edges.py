"""Block GEMM loops on descriptors, operands of any alignment and size: exact against integer
products (small whole numbers: every partial sum is exact)."""

import numpy as np
import pytest

import enceladus_amd as ek
import enceladus_amd.language as tl
from examples.matmul import matmul_desc

pytestmark = pytest.mark.gpu


def whole(rows, cols, seed, lead, dtype="float16"):
    """A [rows, cols] view that starts `lead` elements into its allocation."""
    import torch
    g = torch.Generator().manual_seed(seed)
    flat = torch.randint(-3, 4, (lead + rows * cols,), generator=g).to(getattr(torch, dtype))
    return flat.cuda()[lead:].view(rows, cols)


@pytest.mark.parametrize("tile", [(32, 32, 16, 1), (64, 64, 32, 4), (64, 128, 128, 4),
                                  (128, 128, 64, 4), (256, 128, 64, 8), (256, 256, 64, 8)])
@pytest.mark.parametrize("mnk", [(1, 1, 1), (7, 9, 5), (64, 8, 8), (65, 72, 129), (33, 65, 31),
                                 (130, 257, 200), (300, 500, 502), (257, 130, 1000)])
@pytest.mark.parametrize("lead", [0, 1])
def test_any_size_and_alignment(mnk, tile, lead):
    m, n, k = mnk
    a, b = whole(m, k, 1, lead), whole(k, n, 2, lead, "float16")
    want = (a.double() @ b.double()).cpu()
    bm, bn, bk, nw = tile
    c = matmul_desc(a, b, bm=bm, bn=bn, bk=bk, num_warps=nw)
    assert np.array_equal(c.double().cpu().numpy(), want.numpy())


@pytest.mark.parametrize("tile", [(32, 32, 16, 1), (64, 64, 32, 4), (128, 128, 64, 4),
                                  (256, 128, 32, 8), (128, 32, 16, 4)])
@pytest.mark.parametrize("mnk", [(1, 1, 1), (5, 3, 7), (64, 4, 4), (65, 71, 130), (257, 132, 500)])
@pytest.mark.parametrize("lead", [0, 1])
def test_any_size_and_alignment_fp32(mnk, tile, lead):
    m, n, k = mnk
    a, b = whole(m, k, 1, lead, "float32"), whole(k, n, 2, lead, "float32")
    bm, bn, bk, nw = tile
    c = matmul_desc(a, b, bm=bm, bn=bn, bk=bk, num_warps=nw)
    assert np.array_equal(c.double().cpu().numpy(), (a.double() @ b.double()).cpu().numpy())


@ek.jit
def part_of_k(a_ptr, b_ptr, c_ptr, M, N, K, first, last, BM: tl.constexpr, BN: tl.constexpr,
              BK: tl.constexpr):
    a = tl.make_tensor_descriptor(a_ptr, [M, K], [K, 1], [BM, BK])
    b = tl.make_tensor_descriptor(b_ptr, [K, N], [N, 1], [BK, BN])
    m0 = tl.program_id(0) * BM
    n0 = tl.program_id(1) * BN
    acc = tl.zeros((BM, BN), dtype=tl.float32)
    for k in range(first, last, BK):
        acc = tl.dot(a.load([m0, k]), b.load([k, n0]), acc)
    rm = m0 + tl.arange(0, BM)[:, None]
    rn = n0 + tl.arange(0, BN)[None, :]
    tl.store(c_ptr + rm * N + rn, acc, mask=(rm < M) & (rn < N))


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("bk", [16, 32])
@pytest.mark.parametrize("span", [(0, 1), (0, 32), (0, 33), (0, 96), (16, 97), (5, 70), (64, 64),
                                  (40, 30), (0, 199), (0, 200), (0, 300)])
@pytest.mark.parametrize("k", [200, 199])
def test_steps_of_a_short_tile_cover_no_more_of_k(span, bk, dtype, k):
    """64x64 tiles of few chunks run two steps at once; what no step covers stays out (NaN)."""
    import torch
    m, n = 100, 72
    first, last = span
    end = min(k, first + -(-max(last - first, 0) // bk) * bk)
    a, b = whole(m, k, 1, 0, dtype), whole(k, n, 2, 0, dtype)
    want = a[:, first:end].double() @ b[first:end].double()
    a[:, end:], b[end:] = float("nan"), float("nan")
    a[:, :first], b[:first] = float("nan"), float("nan")
    c = torch.full((m, n), -1.0, device="cuda")
    part_of_k[(2, 2)](a, b, c, m, n, k, first, last, BM=64, BN=64, BK=bk, num_warps=4)
    assert torch.equal(c.double(), want)


@pytest.mark.parametrize("bk", [16, 32, 64])
@pytest.mark.parametrize("first,dma", [(0, True), (16, True), (48, True), (5, False), (8, False),
                                       (12, False)])
def test_k_ranges_of_aligned_operands(first, dma, bk):
    """LDS DMA moves whole 16-byte chunks: only ranges that start on one take it, and their
    merged steps cover no more of k than the program's (NaN beyond); the last elements stay."""
    import torch
    m, n, k = 96, 80, 208
    for last in (first + 1, 100, 160, 207, 208, 300):
        end = min(k, first + -(-max(last - first, 0) // bk) * bk)
        a, b = whole(m, k, 1, 0), whole(k, n, 2, 0)
        want = a[:, first:end].double() @ b[first:end].double()
        a[:, end:], b[end:], a[:, :first], b[:first] = (float("nan"),) * 4
        c = torch.full((m, n), -1.0, device="cuda")
        ck = part_of_k[(2, 2)](a, b, c, m, n, k, first, last, BM=64, BN=64, BK=bk, num_warps=4)
        assert ("ek::GemmDma" in ck.hip) == dma
        assert torch.equal(c.double(), want), (first, last)


@ek.jit
def shifted_columns(a_ptr, b_ptr, c_ptr, M, N, K, BY: tl.constexpr, POINTERS: tl.constexpr,
                    BM: tl.constexpr, BN: tl.constexpr, BK: tl.constexpr):
    m0 = tl.program_id(0) * BM
    n0 = tl.program_id(1) * BN + BY
    rm, rn, rk = m0 + tl.arange(0, BM), n0 + tl.arange(0, BN), tl.arange(0, BK)
    acc = tl.zeros((BM, BN), dtype=tl.float32)
    if POINTERS:
        ap = a_ptr + rm[:, None] * K + rk[None, :]
        bp = b_ptr + rk[:, None] * N + rn[None, :]
        for k in range(0, K, BK):
            a = tl.load(ap, mask=(rm[:, None] < M) & (rk[None, :] + k < K), other=0.0)
            b = tl.load(bp, mask=(rk[:, None] + k < K) & (rn[None, :] < N), other=0.0)
            acc = tl.dot(a, b, acc)
            ap += BK
            bp += BK * N
    else:
        da = tl.make_tensor_descriptor(a_ptr, [M, K], [K, 1], [BM, BK])
        db = tl.make_tensor_descriptor(b_ptr, [K, N], [N, 1], [BK, BN])
        for k in range(0, K, BK):
            acc = tl.dot(da.load([m0, k]), db.load([k, n0]), acc)
    tl.store(c_ptr + rm[:, None] * N + rn[None, :], acc,
             mask=(rm[:, None] < M) & (rn[None, :] < N))


@pytest.mark.parametrize("pointers", [False, True])
@pytest.mark.parametrize("by", [0, 3, 4, 8])
def test_tiles_whose_first_column_starts_no_chunk(by, pointers):
    import torch
    m, n, k = 64, 176, 96
    a, b = whole(m, k, 1, 0), whole(k, n, 2, 0)
    c = torch.full((m, n), -1.0, device="cuda")
    ck = shifted_columns[(1, 3)](a, b, c, m, n, k, BY=by, POINTERS=pointers, BM=64, BN=64, BK=32,
                                 num_warps=4)
    assert ("ek::GemmDma" in ck.hip) == (by % 8 == 0) and "ek::Gemm" in ck.hip
    assert torch.equal(c[:, by:].double(), (a.double() @ b.double())[:, by:])
    assert bool((c[:, :by] == -1).all())
