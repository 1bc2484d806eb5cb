"""The bytes of a row of logits that the sampler's buffer descriptor serves (csrc/row_extent.h):
every id of the row, and nothing that could lie on another page, wherever the row begins."""

import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <stdio.h>
#include "row_extent.h"
using dsv41::row_extent;

// The hardware's range check: a load of `size` bytes at `off` of a buffer of `n` bytes is served
// dword by dword (a smaller load whole).
static bool served(uint32_t off, uint32_t size, uint32_t n) { return off + size <= n; }

int main() {
  for (int esize = 2; esize <= 4; esize += 2)
    for (int V = 1; V < 300; ++V) {
      const uint32_t end = (uint32_t)V * esize;
      // vector loads from a 16-byte boundary: the dword of every id, no dword without one
      const uint32_t n = row_extent(V, esize, true);
      for (uint32_t off = 0; off < end + 64; off += 4)
        if (served(off, 4, n) != (off < end)) return printf("vector V %d esize %d off %u\n", V, esize, off), 1;
      // single loads from any element: every id and none past the row
      const uint32_t m = row_extent(V, esize, false);
      for (uint32_t off = 0; off < end + 64; off += esize)
        if (served(off, esize, m) != (off < end)) return printf("single V %d esize %d off %u\n", V, esize, off), 1;
    }
  return 0;
}
"""


def test_rows_are_served_whole_and_no_further(tmp_path):
    src = tmp_path / "extent.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "extent"
    subprocess.run(["g++", "-std=c++17", "-I", str(ROOT / "tiny-dsv41_amd" / "csrc"), "-o", str(exe), str(src)], check=True)
    got = subprocess.run([str(exe)], capture_output=True, text=True)
    assert got.returncode == 0, got.stdout
