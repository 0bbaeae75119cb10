"""Which masked loads take the clamped path (all of a thread's vectors read at once, those
past the edge from the last selected columns): only masks that select a leading box of a tile
whose rows are contiguous over their whole length."""

import numpy as np
import pytest

import enceladus
import enceladus.language as tl

F = np.zeros(16, np.float32)


@enceladus.jit
def _upper(x_ptr, o_ptr, n, s, BLOCK: tl.constexpr, KIND: tl.constexpr):
    c = tl.arange(0, BLOCK)
    x = x_ptr + tl.program_id(0) * s
    if KIND == "lt":
        v = tl.load(x + c, mask=c < n, other=0.0)
    elif KIND == "gt":
        v = tl.load(x + c, mask=n > c, other=0.0)
    elif KIND == "le":
        v = tl.load(x + c, mask=c <= n, other=0.0)
    elif KIND == "lower":
        v = tl.load(x + c, mask=(c < n) & (c >= 1), other=0.0)
    elif KIND == "or":
        v = tl.load(x + c, mask=(c < n) | (c == 5), other=0.0)
    elif KIND == "strided":
        v = tl.load(x + c * 2, mask=c < n, other=0.0)
    elif KIND == "runs":
        v = tl.load(x + (c // 16) * s + c % 16, mask=c < n, other=0.0)
    elif KIND == "scaled":
        v = tl.load(x + c, mask=c * 2 < n, other=0.0)
    elif KIND == "reversed":
        v = tl.load(x + c, mask=BLOCK - 1 - c < n, other=0.0)
    tl.store(o_ptr + c, v)


@pytest.mark.parametrize("kind,clamped", [
    ("lt", True), ("gt", True), ("le", True), ("lower", False), ("or", False),
    ("strided", False), ("runs", False), ("scaled", False), ("reversed", False)])
def test_which_masks_clamp(kind, clamped):
    src = _upper.warmup(F, F, 781, 783, BLOCK=2048, KIND=kind).hip
    assert ("ek::edge_shift" in src) == clamped
    # the element-wise path stays for boxes narrower than a vector
    assert not clamped or "? *(" in src


def test_unaligned_rows_use_element_aligned_vectors():
    aligned = _upper.warmup(F, F, 784, 784, BLOCK=2048, KIND="lt").hip
    odd = _upper.warmup(F, F, 783, 783, BLOCK=2048, KIND="lt").hip
    assert "ek::vload<float, 4>" in aligned or "ek::vload_nt<float, 4>" in aligned
    assert "ek::vload_u<float, 4>" in odd and "ek::vload_nt" not in odd
