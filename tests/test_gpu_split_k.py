"""Block GEMM loops split along k over several workgroups per tile: exact against integer
products (every partial sum is exact), the same bits on every launch, whole against sliced, on
several streams and threads, and under graph capture (where one workgroup walks the slices)."""

import threading

import numpy as np
import pytest

from enceladus_amd.runtime import compile as C
from examples.matmul import matmul, matmul_desc
from examples.matmul_fused import matmul_bias_gelu
from tests.test_gpu_gemm_edges import whole

pytestmark = pytest.mark.gpu


def _force(monkeypatch, n):
    monkeypatch.setattr(C, "split_factor", lambda split, tiles, hi: n)


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("slices", [1, 2, 3, 5, 16])
@pytest.mark.parametrize("mnk", [(64, 64, 512), (1, 70, 500), (65, 130, 1000), (33, 9, 64)])
def test_sliced_products_are_exact(mnk, slices, dtype, monkeypatch):
    _force(monkeypatch, slices)
    m, n, k = mnk
    a, b = whole(m, k, 1, 0, dtype), whole(k, n, 2, 0, dtype)
    want = (a.double() @ b.double()).cpu().numpy()
    for f, tile in ((matmul_desc, (64, 64, 64)), (matmul, (64, 64, 32))):
        for _ in range(3):           # the tile counters are back at zero after each launch
            c = f(a, b, bm=tile[0], bn=tile[1], bk=tile[2])
            assert np.array_equal(c.double().cpu().numpy(), want)


def test_which_launches_split():
    """Few tiles and a long k split; a grid that fills half of the CUs, or a short k, does not;
    the slices' rows fit the workspace."""
    from enceladus_amd.runtime import hip
    cus = C.coarsen_cap()
    sp = {"hi": 5, "bk": 64, "words": 4096, "step_us": 0.33}
    assert C.split_factor(sp, 16, 8192) > 1
    assert C.split_factor(sp, cus // 2 + 1, 1 << 20) == 1
    assert C.split_factor(sp, 16, 512) == 1 and C.split_factor(sp, 16, 0) == 1
    for tiles in (1, 3, 16, cus // 2):
        for words in (1024, 16384, 65536):
            for hi in (64, 4096, 1 << 24):
                n = C.split_factor(dict(sp, words=words), tiles, hi)
                assert n == 1 or (hip.SPLIT_COUNTERS + n * tiles * words) * 4 <= \
                    hip.WORKSPACE_BYTES
                assert n == 1 or n <= -(-hi // 64) // 2


def test_epilogue_runs_once_and_is_deterministic(monkeypatch):
    import torch
    g = torch.Generator(device="cuda").manual_seed(0)
    a = torch.randn(48, 2048, generator=g, device="cuda").half()
    b = (torch.randn(2048, 200, generator=g, device="cuda") / 45).half()
    bias = torch.randn(200, generator=g, device="cuda").half()
    first = None
    for n in (1, 4):
        _force(monkeypatch, n)
        outs = [matmul_bias_gelu(a, b, bias, bm=64, bn=64, bk=64) for _ in range(4)]
        assert all(torch.equal(o, outs[0]) for o in outs)
        first = outs[0] if first is None else first
        torch.testing.assert_close(outs[0].float(), first.float(), rtol=2e-3, atol=1e-3)


def test_streams_and_threads_have_their_own_workspace(monkeypatch):
    import torch
    _force(monkeypatch, 4)
    a, b = whole(64, 4096, 1, 0), whole(4096, 128, 2, 0)
    want = a.double() @ b.double()
    bad = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(50):
                c = matmul_desc(a, b, bm=64, bn=64, bk=64)
            s.synchronize()
            if not torch.equal(c.double(), want):
                bad.append(1)
    torch.cuda.synchronize()
    ts = [threading.Thread(target=work) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_captured_launches_do_not_split(monkeypatch):
    import torch
    _force(monkeypatch, 4)
    a, b = whole(64, 4096, 1, 0), whole(4096, 128, 2, 0)
    c = torch.empty(64, 128, dtype=torch.float16, device="cuda")
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        matmul_desc(a, b, c, bm=64, bn=64, bk=64)      # compiled and loaded before the capture
    torch.cuda.synchronize()
    want = c.clone()
    g = torch.cuda.CUDAGraph()
    seen = []
    real = C.workspace
    monkeypatch.setattr(C, "workspace", lambda st: seen.append(real(st)) or seen[-1])
    with torch.cuda.graph(g, stream=s):
        matmul_desc(a, b, c, bm=64, bn=64, bk=64)
    assert seen == [0]
    for _ in range(3):
        c.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want)
        matmul_desc(a, b, bm=64, bn=64, bk=64)         # eager work between replays


def _normal(rows, cols, seed, dtype):
    import torch
    g = torch.Generator().manual_seed(seed)
    return torch.randn(rows, cols, generator=g).to(getattr(torch, dtype)).cuda()


@pytest.mark.parametrize("dtype", ["float16", "float32"])
@pytest.mark.parametrize("slices", [2, 3, 7])
@pytest.mark.parametrize("mnk", [(64, 64, 512), (33, 70, 1000), (130, 264, 1024), (5, 3, 999)])
def test_launches_without_a_workspace_have_the_same_bits(mnk, slices, dtype, monkeypatch):
    """One workgroup per tile walks the slices in turn: same sums in the same order."""
    import torch
    m, n, k = mnk
    a, b = _normal(m, k, 1, dtype), _normal(k, n, 2, dtype)
    tiles = [(matmul_desc, 64, 64, 64, 4), (matmul, 64, 64, 32, 4), (matmul_desc, 128, 128, 32, 4)]
    if dtype == "float16":
        tiles.append((matmul_desc, 256, 256, 64, 8))
    for f, bm, bn, bk, nw in tiles:
        outs = []
        for ws in (True, False):
            with monkeypatch.context() as mp:
                mp.setattr(C, "split_factor", lambda split, tiles, hi: slices)
                if not ws:
                    mp.setattr(C, "workspace", lambda stream: 0)
                outs += [f(a, b, bm=bm, bn=bn, bk=bk, num_warps=nw) for _ in range(2)]
        assert all(torch.equal(o, outs[0]) for o in outs), (f.__name__, bm, bn, bk)


@pytest.mark.parametrize("k", [624, 272, 160])
def test_broadcast_rows_without_a_workspace(k, monkeypatch):
    """Rows of B that coincide: the ragged last step, which runs after the loop, ends the last
    slice (10 steps of 64 in slices of 4) or is all of it (5 in slices of 2, 3 in slices of 1)."""
    import torch
    _force(monkeypatch, 3)
    a = _normal(64, k, 1, "float16")
    b = _normal(1, 128, 2, "float16").expand(k, 128)
    want = matmul(a, b)
    torch.testing.assert_close(want.double(), a.double() @ b.double(), rtol=2e-2, atol=2e-2)
    monkeypatch.setattr(C, "workspace", lambda stream: 0)
    assert torch.equal(matmul(a, b), want)


@pytest.mark.parametrize("path", ["warm", "general"])
def test_captured_and_late_streams_have_the_same_bits(path, tmp_path):
    """A shape that the rule splits: eager, captured, and on more streams than have workspaces."""
    import contextlib

    import enceladus
    import torch
    a, b = _normal(64, 4096, 1, "float16"), _normal(4096, 512, 2, "float16") / 64
    bias = _normal(1, 512, 3, "float16")[0]
    out = torch.empty(64, 512, dtype=torch.float16, device="cuda")
    traces = iter(range(100))

    def call(o):
        cm = enceladus.capture(str(tmp_path / f"{next(traces)}.json")) if path == "general" \
            else contextlib.nullcontext()
        with cm:
            return matmul_bias_gelu(a, b, bias, o, bm=64, bn=64, bk=128)
    want = call(torch.empty_like(out))
    assert C.split_factor({"bk": 128, "words": 4096, "step_us": 0.655}, 8, 4096) > 1
    streams = [torch.cuda.Stream() for _ in range(12)]
    torch.cuda.synchronize()
    for s in streams:
        with torch.cuda.stream(s):
            got = call(torch.empty_like(out))
        s.synchronize()
        assert torch.equal(got, want)
    if path == "general":
        return                                      # a dispatch trace waits for each launch
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        call(out)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        call(torch.empty_like(out))


def test_first_split_launch_beside_another_threads_capture(monkeypatch):
    """A stream's workspace is made by its first split launch, also while another thread captures
    (in the global mode, which forbids allocations): neither disturbs the other."""
    import torch
    from enceladus_amd.runtime import hip
    _force(monkeypatch, 4)
    a, b = whole(64, 4096, 1, 0), whole(4096, 128, 2, 0)
    c, d = (torch.zeros(64, 128, dtype=torch.float16, device="cuda") for _ in range(2))
    want = a.double() @ b.double()
    matmul_desc(a, b, c, bm=64, bn=64, bk=64)            # compiled and loaded
    side, own = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    hip.call("ek_workspace_release")                      # no stream has one
    seen, errors = [], []
    real = C.workspace
    monkeypatch.setattr(C, "workspace", lambda st: seen.append(real(st)) or seen[-1])

    def launch():
        try:
            with torch.cuda.stream(own):
                matmul_desc(a, b, d, bm=64, bn=64, bk=64)
        except Exception as e:  # noqa: BLE001
            errors.append(e)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side, capture_error_mode="global"):
        matmul_desc(a, b, c, bm=64, bn=64, bk=64)
        t = threading.Thread(target=launch)
        t.start()
        t.join()
    torch.cuda.synchronize()
    assert not errors and seen[0] == 0 and seen[1] != 0
    assert torch.equal(d.double(), want)
    for _ in range(3):
        c.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(c.double(), want)


def test_the_per_thread_stream_has_no_workspace():
    """hipStreamPerThread is one handle for a stream of each thread, which are not ordered."""
    assert C.workspace(2) == 0


def test_large_accumulators_split_less():
    """One workgroup reads all rows of its tile: 256x256 tiles (256 KB a row) take fewer slices
    than 128x128 ones of the same loop, and none where the unsplit loop is as fast."""
    big, mid = ({"bk": 64, "words": w, "step_us": st} for w, st in ((65536, 1.71), (16384, 0.655)))
    assert C.split_factor(big, 4, 1024) == 1          # 22.8 us unsplit, 27.7 over 2, 34.2 over 5
    assert 2 < C.split_factor(big, 4, 2048) < 6       # 38.7, 34.4 over 3, 54.3 over 10
    assert 4 < C.split_factor(big, 4, 8192) < 10      # 143.9, 58.5 over 8, 74.8 over 15
    assert 4 < C.split_factor(mid, 16, 8192) < 12     # 84.8, 26.8 over 8, 32.9 over 15
    assert C.split_factor(big, 4, -64) == 1
