"""Block GEMM loops over operands whose rows coincide, overlap or descend (row strides of 0,
shorter than the row, negative): exact against integer products of the same views (every partial
sum is exact), through pointer tiles and through descriptors, aligned (LDS DMA) and not."""

import numpy as np
import pytest

import enceladus
import enceladus.language as tl
from examples.matmul import matmul, matmul_kernel

pytestmark = pytest.mark.gpu


@enceladus.jit
def desc_rows(a_ptr, b_ptr, c_ptr, M, N, K, sa, sb, BM: tl.constexpr, BN: tl.constexpr,
              BK: tl.constexpr):
    a = tl.make_tensor_descriptor(a_ptr, [M, K], [sa, 1], [BM, BK])
    b = tl.make_tensor_descriptor(b_ptr, [K, N], [sb, 1], [BK, BN])
    n0, m0 = tl.program_id(0) * BN, tl.program_id(1) * BM
    acc = tl.zeros((BM, BN), dtype=tl.float32)
    for k in range(0, K, BK):
        acc = tl.dot(a.load([m0, k]), b.load([k, n0]), acc)
    rm, rn = m0 + tl.arange(0, BM)[:, None], n0 + tl.arange(0, BN)[None, :]
    tl.store(c_ptr + rm * N + rn, acc.to(c_ptr.dtype.element_ty), mask=(rm < M) & (rn < N))


def rows(n, cols, stride, seed, dtype):
    """(device tensor that starts at the first row, the CPU values) of n rows `stride` apart, in
    an allocation that ends with the last element: NaN lies around the rows."""
    import torch
    span = (n - 1) * abs(stride) + cols
    g = torch.Generator().manual_seed(seed)
    flat = torch.full((span + 64,), float("nan"))
    flat[32:32 + span] = torch.randint(-3, 4, (span,), generator=g).float()
    flat = flat.to(getattr(torch, dtype))
    first = 32 + (span - cols if stride < 0 else 0)
    pick = first + np.arange(n)[:, None] * stride + np.arange(cols)[None, :]
    return flat.cuda()[first:], flat.double().numpy()[pick]


def strides(cols):
    return [0, 16, cols - 16, cols, cols + 24]


SIZES = [(64, 64, 64), (100, 96, 208), (130, 264, 528), (37, 83, 101), (65, 90, 333)]
TILES = [(64, 64, 32, 4), (128, 128, 64, 4), (256, 128, 64, 8)]


def check(mnk, tile, sa, sb, dtype="float16", forms=(True, False)):
    import torch
    m, n, k = mnk
    bm, bn, bk, nw = tile
    a, av = rows(m, k, sa, 1, dtype)
    b, bv = rows(k, n, sb, 2, dtype)
    want = av @ bv
    for pointers in forms:
        c = torch.full((m, n), 7.0, dtype=torch.float32, device="cuda")
        grid = (enceladus.cdiv(n, bn), enceladus.cdiv(m, bm))
        if pointers:
            matmul_kernel[grid](a, b, c, m, n, k, sa, 1, sb, 1, n, 1, BM=bm, BN=bn, BK=bk,
                                num_warps=nw)
        else:
            desc_rows[grid](a, b, c, m, n, k, sa, sb, BM=bm, BN=bn, BK=bk, num_warps=nw)
        assert np.array_equal(c.double().cpu().numpy(), want), (pointers, sa, sb)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("mnk", SIZES)
def test_coinciding_and_overlapping_rows(mnk, tile):
    m, n, k = mnk
    for sa in strides(k):
        for sb in (n, n + 24):
            check(mnk, tile, sa, sb)
    for sb in strides(n):
        check(mnk, tile, k, sb)


def test_broadcast_operands_through_the_wrapper():
    import torch
    m, n, k = 192, 128, 256
    x = torch.randint(-3, 4, (1, k)).half().cuda()
    w = torch.randint(-3, 4, (k, n)).half().cuda()
    want = x.double().expand(m, k) @ w.double()
    assert torch.equal(matmul(x.expand(m, k), w).double(), want)
    y = torch.randint(-3, 4, (1, n)).half().cuda()
    a = torch.randint(-3, 4, (m, k)).half().cuda()
    assert torch.equal(matmul(a, y.expand(k, n)).double(), a.double() @ y.double().expand(k, n))


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("mnk", SIZES)
def test_descending_rows(mnk, dtype):
    """A pointer to the last row in memory and a negative stride (32-bit offsets are unsigned)."""
    m, n, k = mnk
    for tile in TILES[:2]:
        for sa in (-k, -(k + 24), -16, -3):
            check(mnk, tile, sa, n, dtype)
        for sb in (-n, -(n + 24), -16, -3):
            check(mnk, tile, k, sb, dtype)
        check(mnk, tile, -k, -(n + 8), dtype)


@pytest.mark.parametrize("tile", [(32, 32, 32, 4), (64, 64, 32, 8), (32, 64, 64, 8),
                                  (128, 32, 32, 8)])
@pytest.mark.parametrize("mnk", SIZES[:3] + SIZES[4:])
def test_pointer_loops_of_tiles_that_go_through_stages(mnk, tile):
    """Tiles the block GEMM loops do not take: their operands are staged one by one."""
    m, n, k = mnk
    for sa in (0, 16, k - 16, k, -k, -(k + 24), -3):
        check(mnk, tile, sa, n, forms=(True,))
    for sb in (0, 16, n - 16, n + 24, -n, -(n + 24), -3):
        check(mnk, tile, k, sb, forms=(True,))
