"""csrc/loads.h on the CPU: no load that it places can reach memory outside its operand, whether the scalar offset
counts in the bounds check (offset >= size - scalar, unsigned) or not (offset >= size)."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "deciax_amd" / "csrc"
GXX = shutil.which("g++")

PRELUDE = r"""
#include <cstdint>
#include <cstdio>
#include <initializer_list>
#include "loads.h"
// 16 bytes at vector offset v, scalar offset s, of a resource of `size` bytes: reach memory only inside [0, end)
static bool safe(uint32_t v, uint32_t s, uint32_t size, uint64_t end) {
  const bool counted = v < uint32_t(size - s), ignored = v < size;  // passes the check under either reading
  return !(counted || ignored) || (uint64_t)v + s + 16 <= end;
}
static bool blocked(uint32_t v, uint32_t s, uint32_t size) { return !(v < uint32_t(size - s)) && !(v < size); }
#define CHECK(...) do { if (!(__VA_ARGS__)) { std::printf("%s\n", #__VA_ARGS__); return 1; } } while (0)
"""

RING = r"""
int main() {
  // rows of lda elements of 2 bytes, tiles of 64 columns, ring of `stages`: what gemm_ring_kernel issues
  for (int tiles : {1, 2, 5, 17})
    for (int pad : {0, 8, 64})
      for (int rows : {1, 7, 32, 255}) {
        const int lda = tiles * 64 + pad, bytes = rows * lda * 2;
        const uint64_t end = ((uint64_t)(rows - 1) * lda + tiles * 64) * 2;  // the operand's last byte
        for (int t = 0; t < tiles + 8; ++t) {
          const LoadRange r = tile_range(t, tiles, bytes, 128);
          for (int row = 0; row < 256; ++row)
            for (int c = 0; c < 8; ++c) {
              const uint32_t v = row * lda * 2 + c * 16;
              CHECK(safe(v, r.at, r.bytes, end));
              if (t >= tiles || row >= rows) CHECK(blocked(v, r.at, r.bytes));
              else CHECK(v < uint32_t(r.bytes - r.at));
            }
        }
      }
  return 0;
}
"""

SPLIT = r"""
int main() {
  // fp32 rows of ld elements in 16-byte chunks, 16 columns a step, up to 128 rows a tile: linear_split_kernel's loads,
  // of an operand that ends with column k of its last row
  for (int k : {64, 68, 100, 1024, 1028})
    for (int64_t pad : {(int64_t)0, (int64_t)4, (int64_t)(1 << 20) - k})
      for (int rows : {1, 7, 127, 128}) {
        const int64_t ld = k + pad;
        const int bytes = (int)(((rows - 1) * ld + k) * 4);
        for (int kk = 0; kk < k; kk += 16)
          for (int64_t row = 0; row < 128; ++row)
            for (int c = 0; c < 4; ++c) {
              const int64_t v = (row * ld + 4 * c) * 4 + column_offset(kk + 4 * c, k, kk * 4);
              CHECK(v < ((int64_t)1 << 31));
              CHECK(safe((uint32_t)v, 0, bytes, bytes));
              if (row >= rows || kk + 4 * c >= k) CHECK(blocked((uint32_t)v, 0, bytes));
              else CHECK(v + 16 <= bytes);
            }
      }
  return 0;
}
"""


@pytest.mark.skipif(GXX is None, reason="no g++")
@pytest.mark.parametrize("name,body", [pytest.param("ring", RING, id="ring"), pytest.param("split", SPLIT, id="split")])
def test_loads_stay_inside_their_operand(tmp_path: Path, name: str, body: str) -> None:
    src, exe = tmp_path / f"{name}.cpp", tmp_path / name
    src.write_text(PRELUDE + body)
    subprocess.run([GXX, "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
