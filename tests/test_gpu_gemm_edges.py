"""Block GEMM loops on descriptors, operands of any alignment and size: exact against integer
products (small whole numbers: every partial sum is exact)."""

import numpy as np
import pytest

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
