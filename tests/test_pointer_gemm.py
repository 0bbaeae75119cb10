"""Which pointer-and-mask loops become descriptor loops (CPU: the IR the pass leaves)."""

import numpy as np
import pytest

import enceladus
import enceladus.language as tl
from enceladus_amd.compiler import ir

H = np.zeros(16, np.float16)


@enceladus.jit
def _loop(a_ptr, b_ptr, c_ptr, M, N, K, sa, sb, sk, KIND: tl.constexpr, BM: tl.constexpr,
          BN: tl.constexpr, BK: tl.constexpr):
    pm, pn = tl.program_id(1), tl.program_id(0)
    rm = pm * BM + tl.arange(0, BM)
    if KIND == "swizzled":
        rm = (pm // 2) * BM - BM + tl.arange(0, BM)
    rn = pn * BN + tl.arange(0, BN)
    rk = tl.arange(0, BK)
    ap = a_ptr + rm[:, None] * sa + rk[None, :] * sk
    bp = b_ptr + rk[:, None] * sb + rn[None, :]
    acc = tl.zeros((BM, BN), dtype=tl.float32)
    if KIND == "trips":
        for k in range(0, tl.cdiv(K, BK)):
            a = tl.load(ap, mask=(rm[:, None] < M) & (rk[None, :] < K - k * BK), other=0.0)
            b = tl.load(bp, mask=(rk[:, None] < K - k * BK) & (rn[None, :] < N), other=0.0)
            acc = tl.dot(a, b, acc)
            ap += BK * sk
            bp += BK * sb
    elif KIND == "computed":
        for k in range(0, K, BK):
            a = tl.load(a_ptr + rm[:, None] * sa + (k + rk)[None, :] * sk,
                        mask=(rm[:, None] < M) & ((k + rk)[None, :] < K), other=0.0)
            b = tl.load(b_ptr + (k + rk)[:, None] * sb + rn[None, :],
                        mask=((k + rk)[:, None] < K) & (rn[None, :] < N), other=0.0)
            acc = tl.dot(a, b, acc)
    elif KIND == "unmasked":
        for k in range(0, K, BK):
            acc = tl.dot(tl.load(ap), tl.load(bp), acc)
            ap += BK * sk
            bp += BK * sb
    else:
        for k in range(0, K, BK):
            ma = (rm[:, None] < M) & (rk[None, :] + k < K)
            mb = (rk[:, None] + k < K) & (rn[None, :] < N)
            if KIND == "a_only":
                b = tl.load(bp, mask=rn[None, :] < N, other=0.0)
            elif KIND == "other":
                b = tl.load(bp, mask=mb, other=1.0)
            else:
                b = tl.load(bp, mask=mb, other=0.0)
            if KIND == "lower":
                a = tl.load(ap, mask=ma & (rm[:, None] >= 3), other=0.0)
            elif KIND == "shrinking":
                a = tl.load(ap, mask=(rm[:, None] + k < M) & (rk[None, :] + k < K), other=0.0)
            else:
                a = tl.load(ap, mask=ma, other=0.0)
            acc = tl.dot(a, b, acc)
            if KIND == "half_step":
                ap += (BK // 2) * sk
            else:
                ap += BK * sk
            bp += BK * sb
    cp = c_ptr + rm[:, None] * N + rn[None, :]
    tl.store(cp, acc.to(tl.float16), mask=(rm[:, None] < M) & (rn[None, :] < N))


LIFTED = ["plain", "trips", "computed", "unmasked", "swizzled"]
KEPT = ["a_only", "other", "lower", "shrinking", "half_step"]


def _ops(kind, dtype=H, sk=1, bm=64, bk=32):
    f = _loop.ir(dtype, dtype, dtype, 100, 90, 70, 71, 91, sk, KIND=kind, BM=bm, BN=64, BK=bk)
    return [op.name for op in ir.walk(f.body)]


@pytest.mark.parametrize("kind", LIFTED + KEPT)
def test_which_loops_are_lifted(kind):
    names = _ops(kind)
    assert (names.count("desc_load") == 2) == (kind in LIFTED)
    assert (names.count("load") == 0) == (kind in LIFTED)


def test_strided_k_and_small_tiles_stay():
    assert "desc_load" in _ops("plain", dtype=np.zeros(16, np.float32))
    assert "desc_load" not in _ops("plain", sk=2)
    assert "desc_load" not in _ops("plain", bm=16)


@pytest.mark.parametrize("tile", [(256, 128, 128, 8), (128, 64, 256, 4), (32, 128, 256, 8),
                                  (64, 256, 256, 8), (256, 256, 128, 8)])
@pytest.mark.parametrize("mnk", [(1000, 3000, 2000), (1024, 1024, 1024)])
def test_tiles_whose_stages_do_not_fit_stay(tile, mnk):
    """Two LDS stages of these tiles are past 160 KB: the loops keep their pointer loads and
    compile, as they do without the rewrite."""
    from examples.matmul import matmul_kernel
    (bm, bn, bk, nw), (m, n, k) = tile, mnk
    args = (H, H, H, m, n, k, k, 1, n, 1, n, 1)
    meta = dict(BM=bm, BN=bn, BK=bk, num_warps=nw)
    names = [op.name for op in ir.walk(matmul_kernel.ir(*args, **meta).body)]
    assert "desc_load" not in names and names.count("load") == 2
    assert matmul_kernel.warmup(*args, **meta).lds_bytes <= 160 * 1024


def test_tiles_whose_stages_fit_are_lifted():
    from examples.matmul import matmul_kernel
    for bm, bn, bk, nw in ((64, 64, 256, 4), (256, 256, 64, 8), (128, 128, 128, 4)):
        names = [op.name for op in ir.walk(matmul_kernel.ir(
            H, H, H, 1000, 3000, 2000, 2000, 1, 3000, 1, 3000, 1, BM=bm, BN=bn, BK=bk,
            num_warps=nw).body)]
        assert names.count("desc_load") == 2


@enceladus.jit
def _stored_by_tile(a_ptr, b_ptr, c_ptr, t_ptr, M, N, K, sa, KIND: tl.constexpr,
                    BM: tl.constexpr, BN: tl.constexpr, BK: tl.constexpr):
    """B in blocks of BN columns, [K, BN] each, one after the other, or at places of a table."""
    pn, pm = tl.program_id(0), tl.program_id(1)
    rm, rk, cn = pm * BM + tl.arange(0, BM), tl.arange(0, BK), tl.arange(0, BN)
    ap = a_ptr + rm[:, None] * sa + rk[None, :]
    at = pn * (K * BN)
    if KIND == "table":
        at = tl.load(t_ptr + pn, mask=pn * BN < N, other=0)
    bp = b_ptr + at + rk[:, None] * BN + cn[None, :]
    acc = tl.zeros((BM, BN), dtype=tl.float32)
    for k in range(0, K, BK):
        a = tl.load(ap, mask=(rm[:, None] < M) & (rk[None, :] + k < K), other=0.0)
        b = tl.load(bp, mask=(rk[:, None] + k < K) & ((pn * BN + cn)[None, :] < N), other=0.0)
        acc = tl.dot(a, b, acc)
        ap += BK
        bp += BK * BN
    rn = pn * BN + cn
    tl.store(c_ptr + rm[:, None] * N + rn[None, :], acc,
             mask=(rm[:, None] < M) & (rn[None, :] < N))


@pytest.mark.parametrize("kind", ["blocks", "table"])
def test_operands_stored_by_tile_are_described_tile_by_tile(kind):
    """Only what a program's own mask selects belongs to its tile: its descriptor starts at the
    tile (column 0) and ends with the selected columns, unlike A's, which is the whole operand."""
    f = _stored_by_tile.ir(H, H, np.zeros(4, np.float32), np.zeros(4, np.int32), 100, 90, 70, 70,
                           KIND=kind, BM=64, BN=64, BK=32)
    loads = [op for op in ir.walk(f.body) if op.name == "desc_load"]
    assert len(loads) == 2
    a, b = loads
    assert b.operands[2].op.name == "const" and b.operands[2].op.attrs["value"] == 0
    assert a.operands[1].op.name != "const"


@pytest.mark.parametrize("tile,dtype,mnk,lifted", [
    ((64, 64, 64, 8), "float16", (1024, 1024, 1024), True),     # staged, aligned rows
    ((64, 64, 64, 8), "float16", (1000, 3000, 2000), False),
    ((32, 64, 64, 4), "float16", (1000, 3000, 2000), True),     # wide tiles of long steps
    ((32, 64, 32, 4), "float16", (1000, 3000, 2000), False),
    ((64, 64, 256, 4), "float32", (1024, 1024, 1024), False),   # fp32 loops are not staged
    ((64, 64, 32, 4), "float32", (1000, 3000, 2000), True),     # the block GEMM loops take any
    ((64, 64, 32, 4), "float16", (999, 3001, 2001), True)])
def test_loops_are_lifted_where_that_is_faster(tile, dtype, mnk, lifted):
    from examples.matmul import matmul_kernel
    (bm, bn, bk, nw), (m, n, k) = tile, mnk
    x = np.zeros(16, dtype)
    names = [op.name for op in ir.walk(matmul_kernel.ir(
        x, x, x, m, n, k, k, 1, n, 1, n, 1, BM=bm, BN=bn, BK=bk, num_warps=nw).body)]
    assert ("desc_load" in names) == lifted
