"""Vector accesses at any element alignment and the clamped loads of ragged tiles: every
element of a masked tile (selected or not) and every guard element around the stored rows,
for tiles whose selected width lies around the vector width and the tile width."""

import numpy as np
import pytest

import enceladus
import enceladus.language as tl

pytestmark = pytest.mark.gpu

BLOCK = 2048


@enceladus.jit
def _row_edges(x_ptr, tile_ptr, o_ptr, n, stride_x, stride_o, BLOCK: tl.constexpr):
    row = tl.program_id(0)
    c = tl.arange(0, BLOCK)
    x = tl.load(x_ptr + row * stride_x + c, mask=c < n, other=7)
    tl.store(tile_ptr + row * BLOCK + c, x)
    tl.store(o_ptr + row * stride_o + c, x, mask=c < n)


@enceladus.jit
def _box_edges(x_ptr, tile_ptr, n_rows, n_cols, stride, BM: tl.constexpr, BN: tl.constexpr):
    pm, pn = tl.program_id(0), tl.program_id(1)
    r = pm * BM + tl.arange(0, BM)
    c = pn * BN + tl.arange(0, BN)
    x = tl.load(x_ptr + r[:, None] * stride + c[None, :],
                mask=(r[:, None] < n_rows) & (n_cols > c[None, :]), other=-3.0)
    tl.store(tile_ptr + r[:, None] * (tl.num_programs(1) * BN) + c[None, :], x)


@pytest.mark.parametrize("dtype", ["int8", "float16", "float32", "int64"])
@pytest.mark.parametrize("n", [1, 3, 4, 7, 8, 9, 255, 257, 1023, 1025, 2047, 2048])
def test_row_edges(n, dtype):
    import torch
    rows, lead = 5, 3
    stride = n + 2 if n % 2 else n + 1          # odd: every row starts at another alignment
    dt = getattr(torch, dtype)
    gen = torch.Generator().manual_seed(n)
    flat = torch.randint(-100, 100, (lead + rows * stride,), generator=gen).to(dt).cuda()
    x = flat[lead:]
    tile = torch.zeros(rows, BLOCK, dtype=dt, device="cuda")
    out = torch.full((lead + rows * stride + 16,), 5, dtype=dt, device="cuda")
    _row_edges[(rows,)](x, tile, out[lead:], n, stride, stride, BLOCK=BLOCK)
    host = flat.cpu()[lead:]
    want = torch.full((rows, BLOCK), 7, dtype=dt)
    wout = torch.full_like(out.cpu(), 5)
    for r in range(rows):
        want[r, :n] = host[r * stride:r * stride + n]
        wout[lead + r * stride:lead + r * stride + n] = want[r, :n]
    assert torch.equal(tile.cpu(), want)
    assert torch.equal(out.cpu(), wout)


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("shape", [(1, 1), (16, 64), (17, 65), (33, 127), (15, 70), (40, 131)])
def test_box_edges(shape, dtype):
    import torch
    rows, cols = shape
    stride = cols + 1
    x = torch.randn(rows, stride, generator=torch.Generator().manual_seed(cols)).to(
        getattr(torch, dtype)).cuda()
    grid = (enceladus.cdiv(rows, 16), enceladus.cdiv(cols, 64))
    tile = torch.zeros(grid[0] * 16, grid[1] * 64, dtype=x.dtype, device="cuda")
    _box_edges[grid](x, tile, rows, cols, stride, BM=16, BN=64)
    want = torch.full_like(tile.cpu(), -3.0)
    want[:rows, :cols] = x.cpu()[:, :cols]
    assert torch.equal(tile.cpu(), want)


@enceladus.jit
def _transpose(x_ptr, o_ptr, M: tl.constexpr, N: tl.constexpr):
    r, c = tl.arange(0, M), tl.arange(0, N)
    x = tl.load(x_ptr + r[:, None] * N + c[None, :])
    tl.store(o_ptr + c[:, None] * M + r[None, :], tl.trans(x))


@pytest.mark.parametrize("shape", [(128, 256), (256, 256), (512, 128), (16, 4096)])
@pytest.mark.parametrize("dtype", ["float32", "float16", "int64"])
def test_layout_conversions_larger_than_the_lds(shape, dtype):
    """256 x 256 float32 tiles (256 KB) and wider ones move through LDS in passes."""
    import torch
    m, n = shape
    x = torch.arange(m * n, device="cuda").remainder(2039).to(getattr(torch, dtype)).view(m, n)
    o = torch.zeros(n, m, dtype=x.dtype, device="cuda")
    _transpose[(1,)](x, o, M=m, N=n, num_warps=8)
    assert torch.equal(o, x.t())


@enceladus.jit
def _cyclic(t_ptr, o_ptr, start, n, BLOCK: tl.constexpr):
    i = tl.program_id(0) * BLOCK + tl.arange(0, BLOCK)
    tl.store(o_ptr + i, tl.load(t_ptr + (start + i) % n))


@pytest.mark.parametrize("dtype", ["int8", "float16", "float32"])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 33, 1000, 1023, 1024, 1025, 4099, 100000])
@pytest.mark.parametrize("start", [0, 1, 5000, -1500])
def test_cyclic_loads(n, start, dtype):
    """`table + x % n` (C's remainder) for tiles inside one period, across its end, over many
    periods, and of negative x."""
    import torch
    size, pad = 3 * 1024, n
    table = torch.arange(2 * n + 1).remainder(113).to(getattr(torch, dtype)).cuda()
    out = torch.zeros(size, dtype=table.dtype, device="cuda")
    _cyclic[(3,)](table[pad:], out, start, n, BLOCK=1024)
    x = np.arange(start, start + size)
    want = table.cpu()[torch.from_numpy(pad + np.fmod(x, n))]
    assert torch.equal(out.cpu(), want)
