// Which problems the kernel of fp8_gemm_skinny.hip takes, and with what tiles: pure arithmetic on sizes, so that a host compiler can
// build it and a test can hold it against the measurements, and against the shapes that the kernel's own tests name, without a GPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "../../include/flaggems_amd.h"

namespace fg {

// Up to 128 rows, or tiles for one round of blocks: both operands through LDS in deep stages.
struct SkinnyPlan {
  bool use;
  int cfg;                       // tile and ring (kSkinnyShapes)
  int tiles_n, tiles_m;          // tiles along N, rows of tiles
  int splits, stages_per_split;  // blocks along K, and the 256-byte stages of each
  size_t workspace_bytes;
};

constexpr int64_t skinny_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// LDS of a block: a compute unit's for eight wavefronts, half of it for four
constexpr int skinny_table_bytes(int ring, int waves) {
  const int room = (waves == 8 ? 160 : 80) * 1024 - ring;
  return room < 24 * 1024 ? room : 24 * 1024;
}

// The instantiations, and their measured time in us (4700 problems of 1 to 128 rows, block scales and row / column scales, every
// split: the choice it leads to is 1-3 % slower than the fastest of all on average):
//   start + fullest * stages * (stage + rows * rows share) + bytes / stream + (rounds - 1) * round + (split ? exchange + fullest * part : 0)
// with `fullest` the blocks that the fullest compute unit works through.  Four wavefronts: two blocks on a unit.
struct SkinnyShape {
  int bm, bn, nst, waves;
  float start, stage, rows, stream_mb, round, exchange, part;
};
constexpr SkinnyShape kSkinnyShapes[] = {
    {16, 32, 6, 4, 3.01f, 0.118f, 0.022f, 9.9f, 0.27f, 1.04f, 0.35f},
    {16, 64, 3, 4, 2.93f, 0.185f, 0.029f, 8.9f, 0.45f, 1.48f, 0.31f},
    {16, 128, 4, 8, 3.26f, 0.224f, 0.053f, 8.0f, 1.54f, 0.70f, 1.34f},
    {32, 32, 4, 4, 3.25f, 0.105f, 0.077f, 10.5f, 0.73f, 1.93f, 0.14f},
    {32, 64, 3, 4, 3.45f, 0.182f, 0.081f, 9.1f, 0.33f, 1.63f, 0.44f},
    {32, 128, 3, 8, 3.90f, 0.258f, 0.095f, 8.4f, 2.57f, 1.18f, 1.27f},
    {64, 32, 3, 4, 3.64f, 0.102f, 0.185f, 10.0f, 1.11f, 2.26f, 0.11f},
    {64, 64, 4, 8, 3.85f, 0.215f, 0.205f, 11.3f, 2.73f, 1.52f, 0.94f},
    {64, 128, 3, 8, 4.96f, 0.276f, 0.216f, 8.9f, 4.52f, 2.29f, 1.22f},
    {128, 64, 3, 8, 4.88f, 0.139f, 0.434f, 8.0f, 3.59f, 2.22f, 1.55f},
};
// The same for several rows of tiles (7100 problems of 129 to 1000 rows): the weights come out of HBM once for all rows of tiles, so
// less of the time is the stream and more of it the stages.
constexpr int kSkinnyFirstOfRows = 6;
constexpr SkinnyShape kSkinnyShapesOfRows[] = {
    {64, 32, 3, 4, 4.07f, 0.18f, 0.06f, 7.92f, 1.84f, 1.82f, 0.08f},
    {64, 64, 4, 8, 4.01f, 0.32f, 0.17f, 17.1f, 2.51f, 1.30f, 1.03f},
    {64, 128, 3, 8, 4.89f, 0.41f, 0.29f, 16.0f, 3.65f, 2.76f, 1.21f},
    {128, 64, 3, 8, 5.23f, 0.39f, 0.28f, 23.3f, 3.66f, 2.10f, 1.66f},
};

inline float skinny_cost(const SkinnyShape& sh, int64_t M, int64_t N, int64_t K, int64_t tiles, int64_t per, int64_t splits, int cus) {
  const int64_t blocks = tiles * splits, places = (int64_t)cus * (sh.waves == 4 ? 2 : 1), rounds = skinny_div(blocks, places);
  const float fullest = sh.waves == 4 ? (blocks <= cus ? 1.f : 2.f * (float)rounds) : (float)rounds;
  const float rows = (float)(skinny_div(M, 4) * 4 < sh.bm ? skinny_div(M, 4) * 4 : sh.bm) / (float)sh.bm;
  return sh.start + fullest * (float)per * (sh.stage + rows * sh.rows) + (float)N * (float)K * 1e-6f / sh.stream_mb + (float)(rounds - 1) * sh.round +
         (splits > 1 ? sh.exchange + fullest * sh.part : 0.f);
}

// Whether a block's scales fit beside its ring.
inline bool skinny_table_fits(const SkinnyShape& sh, int64_t stages) {
  const int64_t kbs = 2 * stages, room = skinny_table_bytes(sh.nst * (sh.bm + sh.bn) * 256, sh.waves);
  return (skinny_div((kbs | 1) * sh.bm, 64) * 64 + skinny_div(kbs, 64) * 64) * 4 <= room;
}

// Where this kernel is the faster one (us, the kernels of the other files -> this one, both with their best split; M rows, N x K; `ldw`: bytes
// from one weight row to the next, which decides only where K is not split, so that no workspace depends on it).  Measured on 256 compute
// units, which the lines in M, N and K are for; rounds and splits follow the units that there are.
//  * up to 64 rows, K of 512 to 896: always (28, 4096 x 896: 5.6 -> 4.2; 16, 11584 x 896: 6.0 -> 4.5).
//  * up to 16 rows, K from 1024: unsplit in one round that fills over three quarters of the units; emptier rounds lose (12, 9216 x 5120:
//    12.0 -> 13.2).  What pays depends on the tile, on K and on how far apart the weight's rows lie (`ldw`): 4 or 8 KB apart, the other kernels'
//    blocks meet on few memory channels.  Geometric means over 25600 problems of 1 to 16 rows, by the tile's weight rows:
//     - 128: K = 4096 0.85-0.90 (16, 28672 x 4096: 27.8 -> 22.8; with rows 4224 bytes apart 1.04-1.11: 3, 30656: 21.3 -> 23.8), 8192 from 9
//       rows 0.86-0.98 (1, 30272: 41.0 -> 44.6, row and column scales); from 9 rows, K in between 0.87-0.97 and, row and column scales, below 1920 0.95
//       (2048 to 4095 1.01-1.05).
//     - 64: K = 4096 0.81-0.95 (4, 14848: 14.8 -> 12.6), 8192 0.82-0.96 (row and column scales up to 8 rows 1.00); from 9 rows, block scales to 10240
//       0.76-0.96 (13, 15872 x 2048: 9.1 -> 8.3), past it 0.97 (up to 12 rows 10241 to 10752 and from 12416 on 0.98-1.06: 9, 16128 x 14336: 38.9 ->
//       41.4); row and column scales to 1280 0.87-0.93, to 4096 from 13 rows 0.98 (up to 12 rows 1.00: 10, 15936 x 3584: 12.0 -> 12.7; past it 1.01-1.10).
//     - 32: block scales from 9 rows, to 4096 0.95, to 6144 from 13 rows 0.98 (up to 12 rows 1.00: 9, 6400 x 4480: 8.0 -> 8.3; rows 8 KB apart: 15,
//       6272 x 4096: 8.4 -> 8.9); 8192, and 4096 with block scales, from 13 rows (14, 6976 x 8192: 13.7 -> 13.3) or in a round over 15/16 full (12,
//       8192 x 8192: 16.6 -> 13.5); otherwise 1.00-1.15 (10, 6464 x 8192: 11.7 -> 12.6).
//  * 9 to 16 rows, block scales, K split: long K against up to 1536 weight rows 0.92 (9, 1536 x 14080: 14.7 -> 8.4; 768 and fewer 0.98), past 16384
//    up to 2560 0.85 (13, 1920 x 17664: 13.9 -> 10.1; up to 12 rows only to 1344: 11, 1472 x 19584 10.2 -> 12.2), and 3585 to 4096 0.93 (16, 4096 x 14336: 15.2 -> 13.8; up to 12 rows with a shorter K 0.97,
//    a quarter of them 3-12 % slower).  In between the activations of the decode kernels fit LDS in ranges that fill the units (10, 2112 x 10240: 7.9 -> 9.4;
//    9, 3072 x 9216: +20 %); row and column scales 1.02.
//  * 17 to 32 rows: 36.6 -> 26.3 (32, 7168 x 16384), 32.4 -> 23.4 (32, 28672 x 4096), 23.2 -> 14.5 (32, 8192 x 8192); up to 6144 weight
//    rows the parts of up to 16 rows are ahead in between (20, 3968 x 6272: 8.4 -> 11.1; 17, 4608 x 7168: 12.2 -> 13.4) and where their activations
//    still fit LDS (18, 1344 x 11264: 7.9 -> 8.8).
//  * 33 to 64 rows: 40.7 -> 28.5 (61, 7168 x 16384), 22.8 -> 16.3 (61, 4096 x 14336), 16.8 -> 12.8 (61, 4608 x 7168), 32.9 -> 25.0 (61,
//    28672 x 4096); narrow weights only if they are long or large (64, 1280 x 5120: 4.8 -> 7.7 against sixteen-row parts).
//  * 65 to 128 rows: 20.5 -> 16.5 (96, 4608 x 7168), 28 -> 20.8 (80, 4096 x 14336), 33 -> 23 (80, 14336 x 4096); weights of more than
//    8192 rows with K past 6144 do better on 128 x 128 tiles, as do, with row and column scales, 5121 to 6656 with long K and many rows (117, 5504 x
//    16128: 32.6 -> 35.9; 103, 5824 x 16000: 31.5 -> 33.9) (128, 28672 x 4096: 34.8 -> 34.9; 104, 9664 x 13440 +23 %), and so do weights that one
//    block's scales do not cover in the split that suits them (96, 7168 x 16384: 39 -> 46 in five parts); short K against 3072 to 4096
//    weight rows does better in two parts (104, 3072 x 2048: 9.0 -> 10.0).
//  * 129 to 1000 rows, in one round of blocks: 17.4 -> 13.8 (256, 4096 x 4096), 15.8 -> 12.3 (200, 7168 x 2304), 36.6 -> 31.4 (256, 8192 x 8192,
//    row and column scales), 10.3 -> 5.7 (600, 896 x 896); geometric mean of 3090 problems 0.70.  Two rounds lose (333, 8192 x 8192 +25 %), and so
//    does a longer K against the persistent kernel's tiles shared along K: more than 80 tiles of 128 x 64 (597, 1664 x 5632: 18.3 -> 20.8; 256,
//    5120 x 7552: 24.8 -> 31.2), more than 40 (701, 704 x 14976: 24.4 -> 35.7), more than 160 past 8192 or past 512 rows (512, 4096 x 14336: 46.5 ->
//    73.7; 628, 2112 x 7168: 24.0 -> 28.1; block scales from 7424: 252, 5376 x 7424: 25.6 -> 29.9).  Against few weight rows the parts of up to 16 rows are ahead (192, 512 x 2816: 5.1 -> 7.3; 200, 768 x
//    3840: 7.3 -> 8.9; 200, 832 x 1792: 5.8 -> 6.4; 426, 512 x 1152: 4.5 -> 5.1).
//  * past 1000 rows: up to 2048 with K to 3072 (1280, 1600 x 1024: 14.4 -> 10.1), or to 4608 against 768 weight rows and fewer (geometric mean
//    0.75; 1942, 384 x 5120: 17.9 -> 21.3; wider ones 0.95 with +15 to +27 % in every tenth); past 2048 K to 2560 (0.65 to 0.73; to 5632 0.93,
//    every tenth +15 %).
inline SkinnyPlan plan_skinny(int64_t M, int64_t N, int64_t K, int64_t ldw, bool block_scales, int cus) {
  SkinnyPlan p = {};
  if (M < 1 || M > 4096 || N < (M > 1000 ? 128 : 512) || K < 512 || K % 128 != 0) return p;
  const int64_t stages = (K / 128 + 1) / 2, bytes = N * K, mb = 1000000;
  int best = -1;
  int64_t best_per = 0;
  const bool narrow_long = block_scales && M > 8 && M <= 16 && ((N <= (M > 12 ? 2560 : 1344) && K > 16384) || (N > 768 && N <= 1536 && K > 9216 && K <= 16384) ||
                                                                (N > 3584 && N <= 4096 && (K >= 14336 || (M > 12 && K > 10240))));
  if (M <= 16 && K >= 1024 && !narrow_long) {
    for (int c = 0; c < 3; ++c) {
      const int64_t tiles = skinny_div(N, (int64_t)kSkinnyShapes[c].bn);
      if (tiles <= cus && tiles * 4 > (int64_t)cus * 3) best = c;
    }
    if (best < 0 || (block_scales && !skinny_table_fits(kSkinnyShapes[best], stages))) return p;
    // the weight's rows lie next to each other; 4 KB apart or a multiple; begin inside a cache line
    const bool own = ldw == K, apart = ldw % 4096 == 0, torn = ldw % 128 != 0;
    const bool full = skinny_div(N, (int64_t)kSkinnyShapes[0].bn) * 16 > (int64_t)cus * 15;
    bool use;
    if (best == 0) {
      use = (own && K % 4096 == 0 && K <= 8192 && (block_scales || K == 8192) && (M > 12 || full)) ||
            (block_scales && M > 8 && K <= (M > 12 ? 6144 : 4096) && (own || ldw % 8192 != 0));
    } else if (best == 1) {
      use = ((apart || torn) && (K == 4096 || (K == 8192 && (block_scales || M > 8)))) ||
            (M > 8 && (block_scales ? M > 12 || K <= 10240 || (K > 10752 && K <= 12288) || K % 4096 == 0 : K <= 1280 || (M > 12 && K <= 4096 && (own || !apart))));
    } else {
      use = ((apart || torn) && (K == 4096 || (K == 8192 && M > 8))) || (M > 8 && ((K > 4096 && K <= 8192) || (!block_scales && K < 1920)));
    }
    if (!use) return p;
    best_per = stages;
  } else {
    bool use = (M <= 64 && K < 1024) || narrow_long;
    const int64_t units = skinny_div(M * N, (int64_t)8192);  // tiles of 128 x 64
    if (M <= 32) use = use || N > 6144 || (N > 4096 && (bytes <= 16 * mb || bytes >= 48 * mb)) || (N > 3072 && bytes >= 40 * mb) || (N >= 1024 && K >= 11008 && M * K >= 240000);
    else if (M <= 64) use = use || N >= 4096 || (N > 3072 && bytes >= 8 * mb) || (N >= 2048 && bytes >= 20 * mb) || (N >= 1536 && K >= 11008);
    else if (M <= 128 && !block_scales && N > 5120 && N <= 6656 && M * K > 1180000) use = false;
    else if (M <= 128) use = N <= 16384 && (N >= 8192 ? K <= 6144 : N > 4096 ? K >= 1024 : N >= 3072 ? K >= 3072 : (N >= 2048 && K >= 6144));
    else if (M <= 1000) use = units <= cus && (K <= 5120 || units <= 40 || (units <= 80 && K <= 8192) || (M <= 512 && K <= (block_scales ? 7168 : 8192) && units > 160)) &&
                              !(M <= 256 && N <= 1024 && bytes <= (N <= 768 ? 6 : 2) * mb) && !(M <= 512 && N <= 512 && bytes <= 2 * mb);
    else use = units <= cus && (M <= 2048 ? K <= 3072 || (K <= 4608 && N <= 768) : K <= 2560);
    if (!use) return p;
    const int first = M <= 16 ? 0 : M <= 32 ? 3 : M <= 64 ? 6 : M <= 128 ? 9 : kSkinnyFirstOfRows, last = M <= 64 ? first + 3 : 10;
    float best_cost = 0.f, any_cost = 0.f;
    bool any_fits = true, one_round = true;
    for (int c = first; c < last; ++c) {
      const SkinnyShape& sh = M > 128 ? kSkinnyShapesOfRows[c - kSkinnyFirstOfRows] : kSkinnyShapes[c];
      const int64_t tiles = skinny_div(N, (int64_t)sh.bn) * skinny_div(M, (int64_t)sh.bm);
      int64_t seen = 0;
      for (int64_t s = 1; s <= 12 && (s == 1 || tiles * s * 2 <= (int64_t)cus * 9); ++s) {
        const int64_t per = skinny_div(stages, s), splits = skinny_div(stages, per);
        if (per == seen || (splits > 1 && (per < 2 || tiles * sh.waves > FG_WORKSPACE_COUNTER_BYTES / 4 ||
                                           tiles * splits * sh.bm * sh.bn * 4 > FG_NOALLOC_SCRATCH_BYTES / 2))) continue;
        seen = per;
        const float cost = skinny_cost(sh, M, N, K, tiles, per, splits, cus);
        const bool fits = !block_scales || skinny_table_fits(sh, per);
        if (any_cost == 0.f || cost < any_cost) { any_cost = cost; any_fits = fits; }
        if (fits && (best < 0 || cost < best_cost)) {
          best = c; best_per = per; best_cost = cost;
          one_round = tiles * splits <= (sh.waves == 4 ? 2 : 1) * (int64_t)cus;
        }
      }
    }
    if (best < 0 || ((M > 64 || (M <= 16 && K >= 1024)) && M <= 128 && !any_fits) || (M > 128 && !one_round)) return p;
  }
  const SkinnyShape& sh = kSkinnyShapes[best];
  p.cfg = best;
  p.tiles_n = (int)skinny_div(N, (int64_t)sh.bn);
  p.tiles_m = (int)skinny_div(M, (int64_t)sh.bm);
  p.stages_per_split = (int)best_per;
  p.splits = (int)skinny_div(stages, best_per);
  const int64_t items = (int64_t)sh.bm * sh.bn / 256 / (sh.waves / 2), own = items > 1 ? items / 2 : 1;
  p.workspace_bytes = p.splits > 1 ? FG_WORKSPACE_COUNTER_BYTES + (size_t)p.tiles_n * p.tiles_m * p.splits * own * sh.waves * 64 * 16 : 0;
  p.use = true;
  return p;
}

}  // namespace fg
