"""The grouped GEMM's grid against its tiles (csrc/grouped_runs.h, compiled for the host):
for every split of M rows into G groups the blocks that the kernel counts for the real
row tiles fit the grid the host sized by M and G alone."""
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "ernie-evolve-results_amd", "csrc")

MAIN = r"""
#include "grouped_runs.h"
#include <cstdio>
#include <random>
#include <vector>
using namespace moe;

int main() {
  std::mt19937 rng(7);
  auto upto = [&](int n) { return (int)(rng() % (unsigned)(n + 1)); };
  long long tried = 0, runs = 0;
  for (int it = 0; it < 200000; ++it) {
    const int G = 1 + upto(255), n_tiles = 1 + upto(40);
    // groups of one kind (fixed sizes at the edges of a row tile) or mixed
    const int kinds[] = {1, 127, 128, 129, 255, 256, 257, 384, 385, 640};
    const int kind = kinds[upto(9)], mode = upto(3);
    std::vector<int> rows(G);
    int M = 0;
    for (int g = 0; g < G; ++g) {
      rows[g] = mode == 0 ? kind : mode == 1 ? (upto(3) ? 0 : kind) : mode == 2 ? upto(300)
                                             : (upto(7) ? upto(20) : upto(2000));
      M += rows[g];
    }
    M += upto(1) * upto(500);  // rows of no group
    if (M == 0) continue;
    int rt = 0, sh = 0;
    for (int r : rows) {
      const int t = (r + 255) / 256;
      rt += t;
      sh += r > 0 && r <= 128;
    }
    for (int log = 0; log < 2; ++log) {  // what the host may have chosen
      const long long grid = (gg_grid(M, G, n_tiles, log) + 7) / 8 * 8;
      for (int KT : {1, 4, 16, 64}) {
        const int l = gg_run(rt, sh, n_tiles, KT, (int)grid);
        if (gg_blocks(rt, sh, n_tiles, l) > grid || (l > log && gg_blocks(rt, sh, n_tiles, 0) > grid)) {
          printf("G=%d M=%d n_tiles=%d rt=%d sh=%d host log=%d: log %d, %d blocks > %lld\n", G, M,
                 n_tiles, rt, sh, log, l, gg_blocks(rt, sh, n_tiles, l), grid);
          return 1;
        }
        runs += l;
        ++tried;
      }
    }
  }
  // n_tiles blocks for each row tile of a long group, its runs for a short one
  for (int n = 1; n < 20; ++n)
    for (int log = 0; log < 2; ++log)
      if (gg_blocks(3, 1, n, log) != 2 * n + (n + (1 << log) - 1) / (1 << log)) return 2;
  printf("ok %lld %lld\n", tried, runs);
  return runs > 0 ? 0 : 3;
}
"""


def test_grid_holds_every_split(tmp_path):
    src = tmp_path / "runs.cpp"
    src.write_text(MAIN)
    exe = str(tmp_path / "runs")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, str(src), "-o", exe],
                   check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.startswith("ok")
