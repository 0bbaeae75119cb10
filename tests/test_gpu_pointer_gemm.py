"""Pointer-and-mask matmul loops on the GPU, rewritten to descriptor loops or not: exact against
integer products and against the general lowering."""

import numpy as np
import pytest

import enceladus
from examples.matmul import matmul
from tests.test_gpu_gemm_edges import whole
from tests.test_pointer_gemm import KEPT, LIFTED, _loop, _stored_by_tile

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [(32, 32, 16, 1), (64, 64, 32, 4), (128, 128, 64, 4),
                                  (256, 256, 64, 8)])
@pytest.mark.parametrize("mnk", [(1, 1, 1), (7, 9, 5), (65, 72, 129), (130, 257, 200),
                                 (300, 500, 502)])
@pytest.mark.parametrize("lead", [0, 1])
def test_pointer_matmul_any_size_and_alignment(mnk, tile, lead):
    m, n, k = mnk
    a, b = whole(m, k, 1, lead), whole(k, n, 2, lead)
    bm, bn, bk, nw = tile
    c = matmul(a, b, bm=bm, bn=bn, bk=bk, num_warps=nw)
    assert np.array_equal(c.double().cpu().numpy(), (a.double() @ b.double()).cpu().numpy())


@pytest.mark.parametrize("kind", LIFTED + KEPT)
@pytest.mark.parametrize("mnk", [(100, 90, 70), (64, 64, 64), (129, 67, 33)])
def test_lifted_loops_match_the_general_lowering(kind, mnk, monkeypatch):
    import torch
    m, n, k = mnk
    # room around both operands: loops without masks read whole blocks
    pad = 64
    a = whole(m + 2 * pad, k + pad, 3, 0)
    b = whole(k + pad, n + pad, 4, 0)
    outs = []
    for mode in ("", "no_pointer_gemm"):
        monkeypatch.setenv("ENCELADUS_CODEGEN", mode)
        c = torch.full((m + 1, n), 9.0, dtype=torch.float16, device="cuda")
        grid = (enceladus.cdiv(n, 64), enceladus.cdiv(m, 64))
        if kind == "swizzled":
            c = torch.full((m + 65, n), 9.0, dtype=torch.float16, device="cuda")
        first = 64 if kind == "swizzled" else 0
        _loop[grid](a[pad:], b, c[first:], m, n, k, k + pad, n + pad, 1, KIND=kind, BM=64,
                    BN=64, BK=32)
        outs.append(c.cpu())
    assert torch.equal(*outs)


@pytest.mark.parametrize("tile", [(256, 128, 128, 8), (32, 128, 256, 8), (256, 256, 128, 8),
                                  (64, 64, 256, 8)])
@pytest.mark.parametrize("mnk", [(130, 257, 200), (256, 128, 512)])
def test_tiles_with_and_without_room_for_two_stages(mnk, tile):
    m, n, k = mnk
    a, b = whole(m, k, 1, 0), whole(k, n, 2, 0)
    bm, bn, bk, nw = tile
    c = matmul(a, b, bm=bm, bn=bn, bk=bk, num_warps=nw)
    assert np.array_equal(c.double().cpu().numpy(), (a.double() @ b.double()).cpu().numpy())


@pytest.mark.parametrize("kind", ["blocks", "table"])
@pytest.mark.parametrize("mnk", [(100, 90, 70), (64, 128, 96), (70, 131, 33), (5, 3, 64)])
def test_operands_stored_by_tile(kind, mnk):
    """Blocks of columns one after the other, with surplus programs past the last one."""
    import torch
    m, n, k = mnk
    bn = 64
    nb = enceladus.cdiv(n, bn)
    a, b = whole(m, k, 1, 0), whole(k, n, 2, 0)
    at = torch.arange(nb).flip(0) if kind == "table" else torch.arange(nb)
    blocks = torch.full((nb, k, bn), float("nan"), dtype=torch.float16, device="cuda")
    for i in range(nb):
        cols = b[:, i * bn:(i + 1) * bn]
        blocks[at[i], :, :cols.shape[1]] = cols
    table = (at * k * bn).to(torch.int32).cuda()
    c = torch.full((m, n), 7.0, device="cuda")
    _stored_by_tile[(nb + 2, enceladus.cdiv(m, 64) + 1)](
        a, blocks, c, table, m, n, k, k, KIND=kind, BM=64, BN=bn, BK=32)
    assert torch.equal(c.double(), a.double() @ b.double())
