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
// The figures are for 16-bit results.  fp32 results with block scales gain as much or more (median 0.6 beyond 32 K-blocks); fp32 and
// fp8 results with row and column scales have the 128-row kernel as their alternative there too: median 0.85 - 0.96 up to four tile
// rows, 0.92 - 1.03 with more (1.08 at worst).
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

// Few rows a group: activation rows a pass of the weight-streaming grouped kernel takes (16, 32 or 64), or 0 where the persistent
// kernel's 64- to 256-row tiles are faster.  The host knows the rows of an average group only; longer groups take several passes,
// which find their weights in a cache.  us, streaming / persistent, groups x [N, K], rows a group:
//   8 x [28672, 4096]: 6: 166 / 202   16: 178 / 198   32: 187 / 219   48: 198 / 238   64: 263 / 238
//   8 x [4096, 14336]: 6:  84 / 112   16:  84 / 113   32:  89 / 111   48:  96 / 117   64: 137 / 120
//   64 x [2048, 4096]: 48: 135 / 142  64: 177 / 144
//   512 x [2048, 4096]: 1: 468 / 2348 (before its table of tile rows)   16: 804 / -   32: 912 / 816   48: 1009 / 869
// With few groups the persistent kernel loses its last round of tiles, with many it does not.  Hence the 24 rows (48 up to 64
// groups), and
//   * large matrices in 32 groups or more: only up to 32 rows, past which its 128-row tiles stop at one a group.  32 x [4096, 14336]:
//     30: 357 / 393   34: 368 / 336   48: 386 / 339; unequal groups (shares falling as the root of the rank) 30: 404 / 440   48: 471 / 402.
//     (26 x [4096, 14336], unequal: 37: 333 / 404; 64 x [2816, 2048]: 48: 92 / 98.)
//   * one or two K-blocks and no more 256-wide tiles than compute units: an item is a single step, and the table of groups in front
//     and the exchange behind it cost 2 - 5 us more than they save, up to about a dozen groups, whose table the persistent kernel
//     scans as quickly.  K = 256: 2 x 7168: 1: 12.7 / 10.5   48: 16.8 / 12.3; 8 x 2048: 1: 13.4 / 11.3.  (K = 384: 2 x 7168: 1: 10.8 / 11.6;
//     K = 256, 16 x 2048: 1: 13.4 / 15.7; 8 x 16384, two rounds: 1: 13.0 / 20.1.)
// A pass of 16 rows streams fastest (4 stages in flight), 32 are 1 - 3 % slower, 64 another 3 - 9 %.  Where one group holds every row
// the passes repeat: 8 x [28672, 4096], 64 rows, 16 a pass 71, 32 a pass 41, persistent 41.  So large matrices, whose passes cost
// most, take 32 rows from 6 a group on, where groups as unequal as routers make them do not lose by it (8 x [4096, 14336], 64 rows:
// 84.6 with 16 a pass and 84.8 with 32 spread evenly, 93 and 88 unequal; 8 x [28672, 4096] with [4096, 14336] behind it, 48 rows: 254
// and 256).  With everything in one group the kernel stays up to 1.9 times slower than the persistent one on large matrices (16 x
// [28672, 4096], 96 rows: 103 / 54; 64 x [4096, 14336], 1024 rows: 253 / 144); spread as routers spread them it is faster.
inline int grouped_stream_pass_rows(int64_t M, int64_t N, int64_t k_blocks, int64_t groups, int64_t cus) {
  const bool large = N * k_blocks * 128 >= 24000000;
  if (k_blocks <= 2 && groups * ((N + 255) / 256) <= cus && groups <= (k_blocks == 1 || M > 24 * groups ? 12 : 8)) return 0;
  if (M <= 16 || M <= (large ? 6 : 8) * groups) return 16;
  if (M <= 24 * groups) return 32;
  if (M <= 32 * groups) return groups <= 64 ? 64 : 0;
  return M <= 48 * groups && groups <= (large ? 31 : 64) ? 64 : 0;
}

// Grouped problems on 256-row tiles whose rows are read through an index: whether the rows are copied into sorted order first.
// Reading through the index costs a block some 6 us at every tile after its first (index loads and their divisions, whose waits
// cover every copy in flight, in two walks); the copy is a launch and moves 2 M K bytes (4096 tokens twice, K = 4096: 12 us).  So not
// where the tiles, with half a tile row left over in every group, make one round only (K up to 1024) or, with a single K-block, two.
// us, read through the index -> copied, groups x [N, K], rows:
//   8 x [28672, 4096], 1118: 320 -> 266, 7825: 1201 -> 918; 6 x [4096, 1024], 4071: 56.7 -> 50.6; 3 x [12800, 4096], 782, one round: 82.1 -> 71.8
//   8 x [7168, 256], 1139: 20.9 -> 24.0; 6 x [1408, 128], 8325: 19.9 -> 23.2; 2 x [3456, 128], 8229: 29.2 -> 31.3
// Of 1000 random problems that the rule takes it makes 0.85 on average, and five are slower by more than 3 %.  The copy lies in the
// workspace: at most 1 GiB.
inline bool gather_copy_pays(int64_t M, int64_t N, int64_t K, int64_t groups, int64_t cus) {
  if (M * K > ((int64_t)1 << 30)) return false;
  const int64_t columns = (N + 255) / 256, bound = M / 256 + groups < M ? M / 256 + groups : M;
  const int64_t half_tiles = (M / 128 + groups) * columns;  // two for every tile of 256 x 256
  if ((K <= 1024 && half_tiles <= 2 * cus) || (K < 256 && half_tiles * 5 <= cus * 22)) return false;
  return (double)(bound * columns) / (double)cus * 6.0 > 5.0 + (double)M * (double)K * 2 / 5e6;
}

// Parts of up to 16 rows in which the decode kernels take 17..512 rows of a lone problem (measurements at the call): two, four,
// eight ... parts of `rows` rows each (three, five and six were measured and are 20-60 % slower than the next power of
// two), fewer where the rows run out before the parts do; the last part starts `back` rows early so that it ends with the last
// row, and the rows it shares with the part before are computed alike by both.
struct DecodeParts {
  int64_t parts, rows, back;  // parts == 0: not taken
};
inline DecodeParts decode_parts(int64_t M, int64_t N, int64_t K) {
  DecodeParts d = {0, 0, 0};
  const int64_t bytes = N * K;
  if (M > 16 && M <= 32 && N <= 6144) d.parts = 2;
  else if (M > 32 && M <= 64 && N <= 8192 && (bytes <= ((int64_t)13 << 20) || (N <= 3072 && bytes <= ((int64_t)26 << 20)))) d.parts = 4;
  else if (M > 64 && M <= 128 && N <= 4096 && bytes <= ((int64_t)23 << 19)) d.parts = 8;
  // (sixteen and thirty-two parts against the very smallest weights; us at M = 129 / 192 / 256, four 64-row parts on the
  // staged-activation kernel -> sixteen parts: N = 512, K = 7168: 11.1 / 11.7 / 11.8 -> 7.8 / 8.0 / 8.6; N = 256, K = 8192: 10.8 / 11.3 / 11.9 ->
  // 5.9 / 6.2 / 8.2; N = K = 1024: 7.1 / 7.4 / 7.5 -> 5.0 / 5.0 / 5.1; not N = 1024, K = 4096: 9.5 -> 10.0; M = 257 / 512 in thirty-two:
  // N = 256, K = 8192: 11.9 / 12.3 -> 8.2 / 9.8; N = K = 1024: 7.5 / 7.6 -> 5.9 / 6.6)
  else if (M > 128 && M <= 256 && (bytes <= ((int64_t)2 << 20) || (N <= 768 && bytes <= ((int64_t)6 << 20)))) d.parts = 16;
  else if (M > 256 && M <= 512 && N <= 4096 && bytes <= ((int64_t)2 << 20)) d.parts = 32;
  else return d;
  d.rows = (M + d.parts - 1) / d.parts;  // <= 16: M <= 16 * parts
  // as many parts as have a row of their own: only the last one is moved back, so the one before has to end inside the matrix
  // (M = 130 in sixteen parts of nine: the fifteenth would end at row 135)
  d.parts = (M + d.rows - 1) / d.rows;
  d.back = d.parts * d.rows - M;  // < rows: rows that the last part shares with the one before
  return d;
}

}  // namespace fg
