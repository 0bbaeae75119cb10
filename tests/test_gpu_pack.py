"""Flat programs of which a workgroup runs several: every element and the guard after it, for
grids around whole workgroups, tiles inside and across the end, cyclic operands of any period,
through warm, cold, timed and captured launches."""

import numpy as np
import pytest

import enceladus
import enceladus.language as tl

pytestmark = pytest.mark.gpu


@enceladus.jit
def _flat(x_ptr, b_ptr, o_ptr, n, period, BLOCK: tl.constexpr):
    i = tl.program_id(0) * BLOCK + tl.arange(0, BLOCK)
    m = i < n
    x = tl.load(x_ptr + i, mask=m)
    b = tl.load(b_ptr + i % period, mask=m)
    tl.store(o_ptr + i, x + b, mask=m)


@enceladus.jit
def _reduce_rows(x_ptr, o_ptr, n, BLOCK: tl.constexpr):
    i = tl.program_id(0) * BLOCK + tl.arange(0, BLOCK)
    x = tl.load(x_ptr + i, mask=i < n, other=0.0)
    tl.store(o_ptr + i, x + tl.sum(x.to(tl.float32), axis=0), mask=i < n)


def _case(n, period, dtype):
    import torch
    g = torch.Generator().manual_seed(n + period)
    dt = getattr(torch, dtype)
    x = torch.randint(-50, 50, (n,), generator=g).to(dt)
    b = torch.randint(-10, 10, (period,), generator=g).to(dt)
    want = x + b[torch.arange(n) % period]
    return x.cuda(), b.cuda(), torch.full((n + 9,), 3, dtype=dt, device="cuda"), want


@pytest.mark.parametrize("dtype", ["int8", "float16", "bfloat16", "float32"])
@pytest.mark.parametrize("period", [1, 15, 16, 99, 1000, 1024, 4099, 10000])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 2048, 4096, 4097, 20003])
def test_packed_programs(n, period, dtype):
    import torch
    x, b, o, want = _case(n, period, dtype)
    src = _flat.warmup(x, b, o, n, period, BLOCK=1024).hip
    assert ("ek_np_x" in src) == (dtype != "float32")      # 16 bytes a thread stay unpacked
    for extra in (0, 1, 3):                                # programs past the end do nothing
        o.fill_(3)
        _flat[(enceladus.cdiv(n, 1024) + extra,)](x, b, o, n, period, BLOCK=1024)
        got = o.cpu()
        assert torch.equal(got[:n], want) and bool((got[n:] == 3).all())


def test_other_launch_paths(tmp_path):
    import torch
    from enceladus_amd.runtime import timing
    x, b, o, want = _case(5000, 99, "float16")
    launch = lambda: _flat[(5,)](x, b, o, 5000, 99, BLOCK=1024)  # noqa: E731
    launch()

    def check():
        torch.cuda.synchronize()
        assert torch.equal(o.cpu()[:5000], want)
        o.fill_(3)
    check()
    with timing.DispatchTimer() as t:
        launch()
    assert t.ms() > 0 and t.count == 1
    check()
    with enceladus.capture(str(tmp_path / "trace.json")):     # the general launch path
        launch()
    check()
    hx, hb, ho = x.cpu().numpy(), b.cpu().numpy(), np.zeros(5000, np.float16)
    _flat[(5, 1, 1)](hx, hb, ho, 5000, 99, BLOCK=1024)
    assert np.array_equal(ho, want.numpy())
    _flat[(5, 2)](x, b, o, 5000, 99, BLOCK=1024)              # an unused second axis repeats
    check()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        launch()
    for _ in range(3):
        g.replay()
        check()
        launch()
        check()


def test_programs_that_reduce_stay_unpacked():
    x = np.zeros(2048, np.float16)
    assert "ek_np_x" not in _reduce_rows.warmup(x, x, 2048, BLOCK=1024).hip


@enceladus.jit
def _reads_back(p_ptr, q_ptr, o_ptr, n, BLOCK: tl.constexpr):
    i = tl.program_id(0) * BLOCK + tl.arange(0, BLOCK)
    m = i < n
    x = tl.load(p_ptr + i, mask=m)
    tl.store(p_ptr + i, x + x, mask=m)
    y = tl.load(q_ptr + i, mask=m)
    tl.store(o_ptr + i, y + y, mask=m)


@pytest.mark.parametrize("dtype", ["int8", "float16"])
@pytest.mark.parametrize("aliased", [False, True])
@pytest.mark.parametrize("n", [1024, 2048, 5000])
def test_programs_that_read_what_they_stored(n, aliased, dtype):
    """Loads stay behind the stores before them, through the same or another argument."""
    import torch
    p = torch.arange(n).remainder(15).to(getattr(torch, dtype)).cuda()
    q = p if aliased else p + 1
    o = torch.zeros_like(p)
    want_o = 4 * p if aliased else 2 * q
    want_p = 2 * p
    _reads_back[(enceladus.cdiv(n, 1024),)](p, q, o, n, BLOCK=1024)
    assert torch.equal(p, want_p) and torch.equal(o, want_o)


def test_programs_that_load_after_a_store_stay_unpacked():
    x = np.zeros(2048, np.float16)
    assert "ek_np_x" not in _reads_back.warmup(x, x, x, 2048, BLOCK=1024).hip
