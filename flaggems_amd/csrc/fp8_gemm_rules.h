// Where the dispatch of the fp8 GEMMs hands over from one kernel to another: pure arithmetic on sizes, so that a host
// compiler can build it and a test can hold it against the measurements without a GPU.
#pragma once

#include <stdint.h>

namespace fg {

// 256 x 128 tiles with three stages, for a lone problem with more 128-row tiles than compute units but no more 256-row ones (so
// over half of the units get one): one round.  The alternatives are two blocks of 128-row tiles on some units (K of up to 32
// K-blocks), and the persistent kernel's 256 x 256 tiles, cut along K and put together through the workspace.  us, alternative ->
// these tiles, from 6100 shapes a mode (M = 129 .. 4096; geometric mean over those that the rule takes: 0.90 with block scales, 0.91
// where they are powers of two, 0.69 and 0.66 with row and column scales on fp8 and int8 operands):
//   block scales: M = 2048, N = K = 4096: 47.1 -> 42.0; M = 1000, N = 7168, K = 2304: 28.4 -> 26.3; M = 3000, N = 2112, K = 7168: 69.7 -> 62.5
//   row and column scales: M = 500, N = 10240, K = 8192: 92.8 -> 70.5; M = 2000, N = 4096, K = 7168: 75.6 -> 59.5
// What it leaves out:
//   * block scales, K-blocks up to 16: with one tile row (M <= 256) the weights are read once instead of twice (M = 256, N = 24576,
//     K = 1536: 25.5 -> 22.4), otherwise there is little to gain, and with few more 128-row tiles than units the second block on a
//     unit costs little: M = 315, N = 10944, K = 1152 (258 tiles): 14.3 -> 16.7; M = 4048, N = 1088, K = 1024 (288): 14.2 -> 15.6.
//   * more than 32 K-blocks on few units, which the persistent kernel's cuts fill: M = 1000, N = 4608, K = 7168 (144 tall tiles): 58.5 -> 59.9;
//     with block scales and more than 56, on up to 160 where it can halve K: M = 512, N = 10240, K = 8192: 66.2 -> 70.6 (K = 7808, 61
//     K-blocks, M = 184, N = 20224: 89.7 -> 67.1).
//   * row and column scales, K-blocks up to 32: the 128-row kernel is quicker there (M = 312, N = 10944, K = 1408: 16.3 -> 21.0; M = 1500,
//     N = 7168, K = 2304: 7 % and more), but where the weights set the time: up to two tile rows and enough K (M = 136, N = 28672, K = 4096:
//     45.0 -> 40.4; M = 479, N = 11648, K = 4096: 43.0 -> 38.5; but M = 200, N = 16832, K = 2176, 264 tiles: 24.7 -> 26.7).
//   * four K-blocks (M = 256, N = 20480, K = 512: 11.9 -> 12.3), and more than 64, which nobody measured.
// Split along K such tiles lose to 128-row ones (M = 256: N = K = 8192 in four: 36.5 -> 41.4): twice the partial sums.
inline bool tall_tiles_pay(bool block_scales, int64_t M, int64_t N, int64_t k_blocks, int64_t cus) {
  if (M <= 128 || k_blocks < 8 || k_blocks > 64) return false;
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), tall = ((M + 255) / 256) * ((N + 127) / 128);
  if (tiles <= cus || tall > cus) return false;
  if (k_blocks > 32) return block_scales && k_blocks > 56 && k_blocks % 2 == 0 ? tall * 8 > cus * 5 : tall * 10 >= cus * 6;
  const bool many = tiles * 20 > cus * 23;
  if (block_scales) return k_blocks > 16 || M <= 256 || many;
  return M <= 256 ? k_blocks > (many ? 16 : 20) : M <= 512 && k_blocks > 24 && many;
}

}  // namespace fg
