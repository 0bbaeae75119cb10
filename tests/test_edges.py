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


_SHIFTS = """
#include <cstdint>
#include <cstdio>
#include <cstring>
#define EK_INLINE inline
static inline uint64_t __builtin_amdgcn_ballot_w64(bool b) { return b; }
namespace ek {
%s
}
template <typename T, int V> int check() {
  int bad = 0;
  T v[V], o[V], w[2 * V];
  for (int i = 0; i < V; ++i) { v[i] = (T)(3 * i + 1); o[i] = (T)(200 - 5 * i); }
  for (int s = 0; s <= V + 1; ++s) {
    T got[V];
    std::memcpy(got, v, sizeof(v));
    ek::edge_shift<T, V>(got, s, o);
    for (int i = 0; i < V; ++i) bad += got[i] != (s < V && i + s < V ? v[i + s] : o[i]);
  }
  std::memcpy(w, v, sizeof(v));
  std::memcpy(w + V, o, sizeof(o));
  for (int s = 0; s < V; ++s) {
    T got[V];
    std::memcpy(got, v, sizeof(v));
    ek::wrap_shift<T, V>(got, s, o);
    for (int i = 0; i < V; ++i) bad += got[i] != w[i + s];
  }
  if (bad) std::printf("%%d-byte elements, %%d a vector: %%d wrong\\n", (int)sizeof(T), V, bad);
  return bad;
}
int main() {
  return (check<uint8_t, 2>() + check<uint8_t, 4>() + check<uint8_t, 8>() + check<uint8_t, 16>() +
          check<uint16_t, 2>() + check<uint16_t, 4>() + check<uint16_t, 8>() +
          check<uint32_t, 2>() + check<uint32_t, 4>() + check<uint64_t, 2>()) != 0;
}
"""


def test_vector_shifts_against_an_element_model(tmp_path):
    """`edge_shift` and `wrap_shift` for vectors of 2, 4, 8 and 16 bytes, compiled for the host
    from the device header's text."""
    import pathlib
    import shutil
    import subprocess
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    header = pathlib.Path(enceladus.__file__).parent.parent / "enceladus_amd" / "csrc" / \
        "include" / "enceladus_cdna4.h"
    text = header.read_text()
    part = text[text.index("template <int N> struct bits_of"):]
    part = part[:part.index("// ----")]
    src = tmp_path / "shifts.cpp"
    src.write_text(_SHIFTS % part)
    subprocess.run(["g++", "-std=c++17", "-w", "-O1", "-o", str(tmp_path / "shifts"), str(src)],
                   check=True)
    r = subprocess.run([str(tmp_path / "shifts")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
