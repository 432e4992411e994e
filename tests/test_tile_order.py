"""The order in which the tiles of a large product are dealt out: every tile of every share to one workgroup, and runs of neighbours that share operands
also where there are very many tokens."""

import subprocess

import pytest

from shrike_amd.csrc.build import CSRC, HIPCC_FLAGS, find_hipcc

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "gemm_bf16.h"
using namespace shk;

int main() {
  // divisions by numbers that the host knows, on both sides of every multiple near either end
  for (unsigned by = 1; by < 70000; by += by < 300 ? 1 : by / 7) {
    const Divisor d = divisor(by);
    for (long long base : {0ll, 65536ll, (1ll << 31) - 1 - 5ll * by})
      for (int m = 0; m < 5; ++m)
        for (int off = -1; off <= 1; ++off) {
          const long long i = (base / by + m) * by + off;
          if (i >= 0 && i < 1ll << 31 && divided(static_cast<int>(i), d) != i / by) return printf("%lld / %u\n", i, by), 1;
        }
    if (divided(2147483647, d) != 2147483647 / static_cast<int>(by)) return printf("the last / %u\n", by), 1;
  }
  const int xs[] = {1, 2, 3, 7, 8, 14, 56, 297}, ys[] = {1, 2, 5, 8, 9, 16, 33, 100};
  for (int x : xs)
    for (int y : ys)
      for (int shares : {1, 2, 3, 7})
        for (int units : {256, 512})
         for (int k : {1024, 4096}) {
          TileOrder order;
          const unsigned groups = big_grid(x, y, shares, 256, 128, k, units, &order);
          std::vector<int> seen(static_cast<size_t>(x) * y * shares, 0);
          for (unsigned g = 0; g < groups; ++g) {
            int tx = -1, ty = -1, share = -1;
            if (!tile_of(order, g, tx, ty, share)) continue;
            if (tx < 0 || tx >= x || ty < 0 || ty >= y || share < 0 || share >= shares) return printf("outside: %d x %d, %d shares\n", x, y, shares), 1;
            ++seen[(static_cast<size_t>(share) * y + ty) * x + tx];
          }
          for (int times : seen)
            if (times != 1) return printf("%d x %d tiles, %d shares: one is dealt out %d times\n", x, y, shares, times), 1;
        }
  // 32 tiles at a time on a die: of 64 x 2,000 or more they are 6 x 6 or so, not 32 x 1
  for (int k : {1024, 4096})
   for (int y : {16, 100, 2000, 2897, 3500, 6000, 20000}) {
    TileOrder order;
    big_grid(64, y, 1, 256, 256, k, 256, &order);
    const int high = (y + order.strips - 1) / order.strips;
    if (high < 4 || high > 8) return printf("64 x %d tiles in %d strips\n", y, order.strips), 1;
  }
  return 0;
}
"""


def test_every_tile_once_and_runs_of_neighbours(tmp_path):
    hipcc = find_hipcc()
    if hipcc is None:
        pytest.skip("no hipcc")
    source, program = tmp_path / "order.hip", tmp_path / "order"
    source.write_text(PROGRAM)
    subprocess.run([hipcc, *HIPCC_FLAGS, f"-I{CSRC}", "--cuda-host-only", str(source), "-o", str(program)], check=True, capture_output=True)
    run = subprocess.run([str(program)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout
