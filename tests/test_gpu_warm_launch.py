"""The warm launch path of coarsened kernels with a second flush kernel: the same counts as the
first (general) launch for every grid shape, on fresh inputs, other streams and grids."""

import numpy as np
import pytest

import enceladus
import enceladus.language as tl

pytestmark = pytest.mark.gpu


@enceladus.jit
def _two_hists(x_ptr, h_ptr, g_ptr, n, NB: tl.constexpr, BLOCK: tl.constexpr):
    pid = tl.program_id(0) + tl.num_programs(0) * tl.program_id(1)
    offs = pid * BLOCK + tl.arange(0, BLOCK)
    b = tl.load(x_ptr + offs, mask=offs < n, other=-1)
    tl.atomic_add(h_ptr + b, 1, mask=(b >= 0) & (b < NB))
    tl.atomic_add(g_ptr + b, 2, mask=(b >= 0) & (b < 7))


@pytest.mark.parametrize("mode", ["", "priv_flush=atomic", "no_privatize"])
def test_warm_histograms(mode, monkeypatch):
    import torch
    monkeypatch.setenv("ENCELADUS_CODEGEN", mode)
    rng = np.random.default_rng(0)
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    for k, (n, grid) in enumerate([(1000, (1,)), (5000, (5,)), (300000, (100, 3)),
                                   (2000000, (2000,)), (5000, (5,)), (1024, (1, 1, 1))]):
        x = rng.integers(0, 50, n).astype(np.int32)
        want = np.bincount(x, minlength=50)[:48]
        t = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
        for s in streams:
            with torch.cuda.stream(s):
                h = torch.zeros(48, dtype=torch.int32, device="cuda")
                g = torch.zeros(7, dtype=torch.int32, device="cuda")
                for _ in range(2):
                    _two_hists[grid](t, h, g, n, NB=48, BLOCK=1024)
            s.synchronize()
            assert np.array_equal(h.cpu().numpy(), 2 * want), (k, mode)
            assert np.array_equal(g.cpu().numpy(), 4 * want[:7]), (k, mode)
