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
