// How many blocks the grouped GEMM's ring kernel has, and how many column tiles each of
// them takes in a row.  Plain C++: the host sizes the grid with it and every block finds
// its tiles with it.
//
// Row tiles are 256 rows.  A short group (at most 128 rows) is a stream of weights; a
// block that takes two column tiles of it in a row starts the second one's loads under
// the first one's end.  The row tiles of longer groups have a block per column tile: they
// share weights, which runs would move apart.
//
// Measured (MI355X, us, one / two tiles a block; weights of N x K): int8, 128 experts,
// 2048 x 512, 4 rows each 41 / 32; bf16, 128 experts, 1024 x 512, 16 rows 30.5 / 27.9;
// bf16, 64 experts, 4096 x 512, 40 rows 56 / 50.  With long K it does not pay, since blocks
// of two tiles leave a longer tail: bf16, 64 experts, 4096 x 2048, 16 rows 195 / 198; the
// two meet at 32 K steps a block.  Four tiles a block: up to 16% faster at 2048 tiles of
// 4 K steps, 14% slower at 512.
#pragma once

namespace moe {

constexpr int kRunFixed = 8;   // start and end of a block, in K steps
constexpr int kRunSteps = 32;  // K steps of a block of two tiles, at most

// Blocks of rt row tiles, sh of them short groups, with 1 << log column tiles a block in
// these.
constexpr int gg_blocks(int rt, int sh, int n_tiles, int log) {
  return (rt - sh) * n_tiles + sh * ((n_tiles + log) >> log);
}

// log: whichever takes the shorter time in rounds of 256 blocks, among the grids of at
// most blocks_max.
constexpr int gg_run(int rt, int sh, int n_tiles, int KT, int blocks_max) {
  const int one = gg_blocks(rt, sh, n_tiles, 0), two = gg_blocks(rt, sh, n_tiles, 1);
  if (one > blocks_max) return 1;
  if (2 * KT > kRunSteps) return 0;
  return ((two + 255) >> 8) * (2 * KT + kRunFixed) <= ((one + 255) >> 8) * (KT + kRunFixed);
}

// The grid for M rows in G groups, with runs of 1 << log in short ones.  q groups that
// have rows take at least the blocks of a short one; the most that rows beyond each
// group's first can add is, without runs, n_tiles for 256 of them, and with runs
// 2 n_tiles - n_tiles / 2 for 256 of them (a group of 257 rows).
constexpr long long gg_grid(int M, int G, int n_tiles, int log) {
  const long long q = G < M ? G : M;
  return q * ((n_tiles + log) >> log) + ((M - q) * n_tiles * (2 + log) + 511) / 512;
}

}  // namespace moe
