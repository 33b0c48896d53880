// Weight-streaming GEMM for few activation rows per weight matrix (up to 64 a pass): expert layers while decoding, where
// hundreds of weight matrices meet one to a few dozen rows each.
//
// Bound: HBM (the weights are read once, 32 .. 128 flops a byte).  Measured, weight bytes of the groups that have rows
// over the launch's time: 512 groups of [2048, 4096], one or two rows each, 5.9 TB/s (the persistent kernel's 64-row tiles:
// 1.2); 8 groups of [28672, 4096], 1 .. 8 rows each, 5.4 - 5.7 TB/s (4.4 - 4.6), 48 rows each 4.8 (4.0); 8 of
// [4096, 14336] 5.2 - 5.6 (3.3 - 4.2).  A copy of 1 GiB moves 4.9 - 5.1 TB/s.  What the design is about is keeping every compute
// unit's queue of weight loads full from the first to the last byte of the launch, whatever the table of groups says.
//
//  * A step is 128 weight rows x 256 bytes of K (two K-blocks) against up to 16 TMX activation rows.  An item is one
//    output piece (group, 128 weight rows, 16 TMX activation rows) = K / 256 steps; the items of all groups that have
//    rows, laid end to end, are cut into one contiguous range of steps per compute unit.  The ranges differ by at most
//    one step, so nothing is left idle by a partly filled last round; a range covers the end of an item, whole items
//    and the beginning of an item.
//  * One block of eight wavefronts per compute unit.  A step's operands travel by global -> LDS copies (256-byte runs:
//    a wavefront instruction covers 4 rows) through a ring of LDS stages, kStages - 1 of them in flight; the ring does
//    not stop at item boundaries: the copies run that many steps ahead of the multiplication, into the next item.  A
//    wavefront copies and multiplies its own 16 weight rows; the activation rows are shared by the block (one barrier a
//    step).
//  * Items shared by several blocks are finished through the workspace, per wavefront: publish the fp32 sums, count in,
//    and whoever arrives last adds all parts in range order (results do not depend on timing) and stores.  A part is
//    8 KB x TMX per block, at most two per block.
//  * The block reads the table of group ends once, in parallel, and keeps (end row, items before) of every group in LDS;
//    walking on to the next item is a few scalar operations then.  (The persistent kernel scans the table in memory at
//    every tile: with 512 groups that was nine tenths of its time.)
//  * Rows gathered through an index: the index entries of the next item are copied to LDS while the current item's
//    operands stream, the routing weights likewise, so an item boundary waits for no load.
//
// LDS images.  A stage holds 128 weight rows of 256 bytes, then the activation rows of 256 bytes; within a row the
// sixteen 16-byte pieces are permuted (physical piece p holds logical piece p ^ (row & 15)), so the 16 rows that a
// wavefront reads together fall into 16 different bank groups.

#include "fp8_gemm_common.h"
#include "fp8_gemm_rules.h"

namespace fg {
namespace {

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kItemCols = 128;               // weight rows of an item, 16 per wavefront
constexpr int kWBytes = kItemCols * 256;     // weight bytes of a step
constexpr int kMaxGroups = 1024;
constexpr int kRing = 8;                     // items whose row indices are kept (the copies run at most 4 items ahead)

struct StreamArgs {
  GemmArgs g;
  // groups: cumulative row ends, forced into ascending order and into [0, M]
  const int* ends;
  int n_groups;
  int64_t w_group_stride, ws_group_stride;
  const int* row_index;  // gather / scatter table, as in PpArgs of the persistent kernel
  int index_div, x_rows; // index_div 0: rows are in order, the table only addresses the results
  int c_rows;
  const float* row_weight;
  int chunks, pairs;     // items per row tile, steps per item
  int min_steps;         // fewest steps worth a block of its own
  float* partials;       // null: items are not shared between blocks
  unsigned int* counters;
};

template <int TMX>
struct Cfg {
  static constexpr int kRows = 16 * TMX;
  static constexpr int kStages = TMX == 1 ? 4 : 3;
  static constexpr int kXBytes = kRows * 256;
  static constexpr int kScaleFloats = 2 * kRows + 64;  // [2][kRows] activation scales, then the two weight scales
  static constexpr int kStageBytes = kWBytes + kXBytes + kScaleFloats * 4;
  static constexpr int kIndexOff = kStages * kStageBytes;           // [kRing][64] row indices
  static constexpr int kWeightOff = kIndexOff + kRing * 64 * 4;     // [kRing][64] row weights
  static constexpr int kTableOff = kWeightOff + kRing * 64 * 4;     // [kMaxGroups + 1] end rows, [kMaxGroups + 1] row tiles before
  static constexpr int kLds = kTableOff + 2 * (kMaxGroups + 2) * 4;
  static constexpr int kXCopies = TMX == 4 ? 2 : 1;                 // copies of activation rows per wavefront and step
  static constexpr int kPerStage = 4 + kXCopies + 1;
  static_assert(kLds <= 160 * 1024, "LDS");
};

// (s_nop 4: the base may have been written by a vector instruction just before, see store_x4_agent)
__device__ __forceinline__ void copy16(uint32_t byte_off, const void* base, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(byte_off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
__device__ __forceinline__ void copy4(uint32_t byte_off, const void* base, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dword %0, %1" : : "v"(byte_off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
template <int PENDING>
__device__ __forceinline__ void wait_copies() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(PENDING) : "memory");
}

// Where a walk stands (uniform): the item's group, its row tile and chunk inside the group, the step inside the item.
struct Walk {
  int group, begin, end;  // rows [begin, end) of the group
  int tile, tiles;        // row tile inside the group
  int chunk, pair;
  int serial;             // items entered so far (selects the ring slot)
};

// Inclusive scans over a wavefront.
__device__ __forceinline__ int wave_scan_max(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d);
    if (lane >= d) v = o > v ? o : v;
  }
  return v;
}
__device__ __forceinline__ int wave_scan_sum(int v, int lane) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int o = __shfl_up(v, d);
    if (lane >= d) v += o;
  }
  return v;
}

template <int TMX>
__global__ __launch_bounds__(kThreads) void fp8_gemm_stream_kernel(StreamArgs a) {
  using C = Cfg<TMX>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const GemmArgs& g = a.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  int* const t_end = reinterpret_cast<int*>(lds + C::kTableOff);
  int* const t_tiles = t_end + kMaxGroups + 2;  // [e]: row tiles of the groups before e; [n_groups]: all of them
  const int E = a.n_groups;

  // ---- the table of groups: ends in ascending order (a running maximum), row tiles before every group (a running sum)
  {
    int* const sums = reinterpret_cast<int*>(lds + C::kIndexOff);  // [2][kWaves], free until the first item
    const int e0 = 2 * tid, e1 = e0 + 1;
    int v0 = e0 < E ? a.ends[e0] : 0, v1 = e1 < E ? a.ends[e1] : 0;
    v0 = v0 < 0 ? 0 : (v0 < g.M ? v0 : g.M);
    v1 = v1 < 0 ? 0 : (v1 < g.M ? v1 : g.M);
    v1 = v1 > v0 ? v1 : v0;
    const int incl = wave_scan_max(v1, lane);
    if (lane == 63) sums[wave] = incl;
    __syncthreads();
    int before = __shfl_up(incl, 1);
    if (lane == 0) before = 0;
    for (int w = 0; w < wave; ++w) before = sums[w] > before ? sums[w] : before;
    v0 = v0 > before ? v0 : before;
    v1 = v1 > v0 ? v1 : v0;
    const int n0 = e0 < E ? (v0 - before + C::kRows - 1) / C::kRows : 0;
    const int n1 = e1 < E ? (v1 - v0 + C::kRows - 1) / C::kRows : 0;
    const int total = wave_scan_sum(n0 + n1, lane);
    if (lane == 63) sums[kWaves + wave] = total;
    __syncthreads();
    int tiles = total - n0 - n1;
    for (int w = 0; w < wave; ++w) tiles += sums[kWaves + w];
    if (e0 < E) { t_end[e0] = v0; t_tiles[e0] = tiles; }
    if (e1 < E) { t_end[e1] = v1; t_tiles[e1] = tiles + n0; }
    if (e0 == E - 1) t_tiles[E] = tiles + n0;
    if (e1 == E - 1) t_tiles[E] = tiles + n0 + n1;
    __syncthreads();
  }

  // ---- this block's range of steps
  const int KP = a.pairs;
  const int items = __builtin_amdgcn_readfirstlane(t_tiles[E]) * a.chunks;
  const int units = a.partials != nullptr ? items * KP : items;  // what the ranges are counted in
  int blocks = a.partials != nullptr ? units / a.min_steps : items;
  blocks = blocks < 1 ? 1 : (blocks < (int)gridDim.x ? blocks : (int)gridDim.x);
  if ((int)blockIdx.x >= blocks || units == 0) return;
  const int q = units / blocks, rem = units - q * blocks;
  const int scale = a.partials != nullptr ? 1 : KP;
  auto range_begin = [&](int b) __attribute__((always_inline)) { return (b * q + (b < rem ? b : rem)) * scale; };
  auto block_of_step = [&](int s) __attribute__((always_inline)) {  // (shared items only: scale is 1)
    const int big = rem * (q + 1);
    return s < big ? s / (q + 1) : rem + (s - big) / q;
  };
  const int lo = range_begin((int)blockIdx.x), hi = range_begin((int)blockIdx.x + 1);
  const int n_steps = hi - lo;

  auto enter_group = [&](Walk& w, int e) __attribute__((always_inline)) {  // the first group from e on that has rows
    int before = __builtin_amdgcn_readfirstlane(t_tiles[e]);
    for (;;) {
      const int after = __builtin_amdgcn_readfirstlane(t_tiles[e + 1]);
      if (after != before || e + 1 >= E) { w.tiles = after - before; break; }
      ++e;
    }
    w.group = e;
    w.begin = e > 0 ? __builtin_amdgcn_readfirstlane(t_end[e - 1]) : 0;
    w.end = __builtin_amdgcn_readfirstlane(t_end[e]);
  };
  auto next_item = [&](Walk& w) __attribute__((always_inline)) {
    w.pair = 0;
    ++w.serial;
    if (++w.tile < w.tiles) return;
    w.tile = 0;
    if (++w.chunk < a.chunks) return;
    w.chunk = 0;
    if (w.group + 1 < E) enter_group(w, w.group + 1);
  };

  // first item of the range: the last group with at most item / chunks row tiles before it
  Walk at;  // the multiplication's walk; the copies have one of their own
  {
    const int item = lo / KP;
    const int row_tile_bound = item / a.chunks;
    int e_lo = 0, e_hi = E - 1;
    while (e_lo < e_hi) {
      const int mid = (e_lo + e_hi + 1) >> 1;
      if (__builtin_amdgcn_readfirstlane(t_tiles[mid]) <= row_tile_bound) e_lo = mid;
      else e_hi = mid - 1;
    }
    at.group = e_lo;
    at.begin = e_lo > 0 ? __builtin_amdgcn_readfirstlane(t_end[e_lo - 1]) : 0;
    at.end = __builtin_amdgcn_readfirstlane(t_end[e_lo]);
    const int before = __builtin_amdgcn_readfirstlane(t_tiles[e_lo]);
    at.tiles = __builtin_amdgcn_readfirstlane(t_tiles[e_lo + 1]) - before;
    const int local = item - before * a.chunks;  // inside the group: chunk by chunk, the row tiles of a chunk together
    at.chunk = local / at.tiles;
    at.tile = local - at.chunk * at.tiles;
    at.pair = lo - item * KP;
    at.serial = 0;
  }
  at.group = __builtin_amdgcn_readfirstlane(at.group);
  at.begin = __builtin_amdgcn_readfirstlane(at.begin);
  at.end = __builtin_amdgcn_readfirstlane(at.end);
  at.tile = __builtin_amdgcn_readfirstlane(at.tile);
  at.tiles = __builtin_amdgcn_readfirstlane(at.tiles);
  at.chunk = __builtin_amdgcn_readfirstlane(at.chunk);
  at.pair = __builtin_amdgcn_readfirstlane(at.pair);
  Walk ahead = at;       // item whose steps are being copied
  Walk beyond = at;      // the item after it

  // ---- copies
  const bool gathered = a.row_index != nullptr && a.index_div > 0;
  const int* const ring_index = reinterpret_cast<const int*>(lds + C::kIndexOff);
  const float* const ring_weight = reinterpret_cast<const float*>(lds + C::kWeightOff);
  const int w_row = lg;                                   // row of a copy's 4 that this lane fetches
  uint32_t w_off[4], x_off[C::kXCopies], s_off = 0;
  const uint8_t *w_base = nullptr, *x_base = nullptr;      // uniform: first byte of the item's rows
  const float* s_base = nullptr;                           // uniform: scales this wavefront copies
  int64_t s_step = 0;
  const bool odd_k = (g.KB & 1) != 0;
  // waves whose copy carries the weight scales: TMX 4 needs two copies for the activation scales (one per K-block)
  const bool ws_wave = TMX == 4 ? (wave & 2) != 0 : (wave & 1) != 0;

  auto copy_index = [&](const Walk& w) __attribute__((always_inline)) {
    if (a.row_index == nullptr) return;
    if (lane < C::kRows) {
      int m = w.begin + w.tile * C::kRows + lane;
      m = m < w.end ? m : w.end - 1;
      copy4((uint32_t)m * 4u, uniform_ptr(a.row_index), lds_base + C::kIndexOff + (uint32_t)((w.serial & (kRing - 1)) * 256));
    }
  };
  // lane-dependent source row of tile row r
  auto source_row = [&](const Walk& w, int r) __attribute__((always_inline)) -> int {
    const int m0 = w.begin + w.tile * C::kRows;
    const int last = w.end - 1 - m0;
    r = r < last ? r : last;
    if (!gathered) return r;
    int src = ring_index[(w.serial & (kRing - 1)) * 64 + r] / a.index_div;
    return src < 0 ? 0 : (src < a.x_rows ? src : a.x_rows - 1);
  };
  auto enter_item = [&](const Walk& w) __attribute__((always_inline)) {  // w: the item whose copies start now
    const int n0 = w.chunk * kItemCols;
    const int m0 = w.begin + w.tile * C::kRows;
    w_base = uniform_ptr(g.W + (int64_t)w.group * a.w_group_stride + (int64_t)n0 * g.ldw);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = j * 4 + w_row;  // row of the wavefront's 16
      int row = wave * 16 + r;
      row = n0 + row < g.N ? row : g.N - 1 - n0;
      w_off[j] = (uint32_t)row * (uint32_t)g.ldw + (uint32_t)((l16 ^ r) << 4);
    }
    x_base = uniform_ptr(g.X + (gathered ? 0 : (int64_t)m0 * g.ldx));
#pragma unroll
    for (int j = 0; j < C::kXCopies; ++j) {
      const int r = TMX == 1 ? wave * 2 + ((lane >> 4) & 1) : (wave * C::kXCopies + j) * 4 + lg;
      x_off[j] = (uint32_t)source_row(w, r) * (uint32_t)g.ldx + (uint32_t)((l16 ^ (r & 15)) << 4);
    }
    if (ws_wave) {
      s_base = uniform_ptr(g.ws + (int64_t)w.group * a.ws_group_stride + (int64_t)w.chunk * g.ws_rs);
      s_off = (uint32_t)(lane & 1) * (uint32_t)g.ws_cs * 4u;
      s_step = g.ws_cs;
    } else {
      s_base = uniform_ptr(g.xs + (gathered ? 0 : (int64_t)m0 * g.xs_rs));
      const int b = TMX == 4 ? (wave & 1) : (lane >> (TMX == 1 ? 4 : 5)) & 1;
      s_off = ((uint32_t)source_row(w, lane & (C::kRows - 1)) * (uint32_t)g.xs_rs + (uint32_t)b * (uint32_t)g.xs_cs) * 4u;
      s_step = g.xs_cs;
    }
    if (a.row_weight != nullptr && lane < C::kRows) {
      int idx = ring_index[(w.serial & (kRing - 1)) * 64 + lane];
      idx = idx < 0 ? 0 : (idx < a.c_rows ? idx : a.c_rows - 1);
      copy4((uint32_t)idx * 4u, uniform_ptr(a.row_weight), lds_base + C::kWeightOff + (uint32_t)((w.serial & (kRing - 1)) * 256));
    }
  };
  auto issue_step = [&](int pair, int slot) __attribute__((always_inline)) {
    const uint32_t stage = lds_base + (uint32_t)(slot * C::kStageBytes);
    const bool half = odd_k && pair == KP - 1;  // the pair's second K-block does not exist: its pieces repeat the first's
    const uint8_t* const wp = uniform_ptr(w_base + (int64_t)pair * 256);
    const uint8_t* const xp = uniform_ptr(x_base + (int64_t)pair * 256);
    const float* const sp = uniform_ptr(s_base + (int64_t)pair * 2 * s_step);
    if (ws_wave) {
      if (lane < 2) copy4(half ? 0u : s_off, sp, stage + kWBytes + C::kXBytes + 2 * C::kRows * 4);
    } else {
      const bool second = TMX == 4 ? (wave & 1) != 0 : lane >= C::kRows;
      const uint32_t off = half && second ? s_off - (uint32_t)g.xs_cs * 4u : s_off;
      if (TMX > 1 || lane < 32) copy4(off, sp, stage + kWBytes + C::kXBytes + (TMX == 4 ? (uint32_t)(wave & 1) * C::kRows * 4 : 0u));
    }
#pragma unroll
    for (int j = 0; j < C::kXCopies; ++j) {
      const int r = TMX == 1 ? wave * 2 + ((lane >> 4) & 1) : (wave * C::kXCopies + j) * 4 + lg;
      const uint32_t off = half && ((l16 ^ (r & 15)) & 8) ? x_off[j] - 128u : x_off[j];
      const uint32_t dst = stage + kWBytes + (uint32_t)(TMX == 1 ? wave * 512 : (wave * C::kXCopies + j) * 1024);
      if (TMX > 1 || lane < 32) copy16(off, xp, dst);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t off = half && ((l16 ^ (j * 4 + w_row)) & 8) ? w_off[j] - 128u : w_off[j];
      copy16(off, wp, stage + (uint32_t)((wave * 4 + j) * 1024));
    }
  };

  // The index entries of item i + 1 are requested when item i is entered.  When item i + 1 is entered they have landed
  // if a step issued after them has (steps land in order); otherwise, with items of very few steps, wait.
  int since_index = 0;
  copy_index(ahead);
  wait_copies<0>();
  enter_item(ahead);
  next_item(beyond);
  const int last_item = (hi - 1) / KP - lo / KP;  // serial of the range's last item
  if (beyond.serial <= last_item) copy_index(beyond);
  int issued = 0, load_slot = 0;
  auto issue_next = [&](bool landed) __attribute__((always_inline)) {  // landed: all but the youngest kStages - 2 steps have
    if (ahead.pair == KP) {
      if (!(landed && since_index >= C::kStages - 1) && a.row_index != nullptr) wait_copies<0>();
      ahead = beyond;
      enter_item(ahead);
      next_item(beyond);
      if (beyond.serial <= last_item) copy_index(beyond);
      since_index = 0;
    }
    issue_step(ahead.pair, load_slot);
    ++ahead.pair; ++issued; ++since_index;
    load_slot = load_slot + 1 == C::kStages ? 0 : load_slot + 1;
  };
#pragma unroll 1
  for (int s = 0; s < C::kStages - 1; ++s)
    if (s < n_steps) issue_next(false);

  v4f acc[TMX];
#pragma unroll
  for (int t = 0; t < TMX; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  int first_pair = at.pair;  // first pair of the current item that this block multiplies
  const int frag_row = l16 * 256;

  for (int s = 0; s < n_steps; ++s) {
    if (n_steps - 1 - s >= C::kStages - 2) wait_copies<(C::kStages - 2) * C::kPerStage>();
    else wait_copies<0>();
    // (a bare barrier: a fence would wait for every copy in flight; the LDS reads of the previous step have returned)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
    if (issued < n_steps) issue_next(true);

    const uint8_t* const sw = lds + slot * C::kStageBytes + wave * 4096 + frag_row;
    const uint8_t* const sx = lds + slot * C::kStageBytes + kWBytes + frag_row;
    const float* const sc = reinterpret_cast<const float*>(lds + slot * C::kStageBytes + kWBytes + C::kXBytes);
    const bool half = odd_k && at.pair == KP - 1;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (b == 1 && half) break;
      auto fragment = [&](const uint8_t* rows) __attribute__((always_inline)) {
        const u32x4 f_lo = *reinterpret_cast<const u32x4*>(rows + (((b * 8 + lg) ^ l16) << 4));
        const u32x4 f_hi = *reinterpret_cast<const u32x4*>(rows + (((b * 8 + 4 + lg) ^ l16) << 4));
        v8i f;
        f[0] = (int)f_lo.x; f[1] = (int)f_lo.y; f[2] = (int)f_lo.z; f[3] = (int)f_lo.w;
        f[4] = (int)f_hi.x; f[5] = (int)f_hi.y; f[6] = (int)f_hi.z; f[7] = (int)f_hi.w;
        return f;
      };
      const v8i wf = fragment(sw);
      const float wsv = sc[2 * C::kRows + b];
#pragma unroll
      for (int t = 0; t < TMX; ++t) {
        const v8i xf = fragment(sx + t * 4096);
        const float f = sc[b * C::kRows + t * 16 + l16] * wsv;
        const v4f p = mfma_fp8_16x16x128(wf, xf, v4f{0.f, 0.f, 0.f, 0.f});
        acc[t][0] = __builtin_fmaf(p[0], f, acc[t][0]);
        acc[t][1] = __builtin_fmaf(p[1], f, acc[t][1]);
        acc[t][2] = __builtin_fmaf(p[2], f, acc[t][2]);
        acc[t][3] = __builtin_fmaf(p[3], f, acc[t][3]);
      }
    }
    slot = slot + 1 == C::kStages ? 0 : slot + 1;

    ++at.pair;
    if (at.pair < KP && s + 1 < n_steps) continue;

    // ---- the item ends here, or the range does
    bool store = true;
    if (!(first_pair == 0 && at.pair == KP)) {
      const int item0 = lo + s - (at.pair - 1);  // first step of the item
      const int fb = block_of_step(item0), lb = block_of_step(item0 + KP - 1);
      const uint32_t lane_off = (uint32_t)lane * 16u;
      constexpr int kPart = TMX * 256;  // floats of one wavefront
      auto part = [&](int b) __attribute__((always_inline)) {
        const int sl = 2 * b + (range_begin(b) > item0 ? 0 : 1);
        return uniform_ptr(a.partials + ((int64_t)sl * kWaves + wave) * kPart);
      };
      float* const mine = part((int)blockIdx.x);
#pragma unroll
      for (int t = 0; t < TMX; ++t) store_x4_agent(mine + t * 256, lane_off, acc[t]);
      wait_copies<0>();
      unsigned int* const cnt = a.counters + fb * kWaves + wave;
      unsigned int prev = 0;
      if (lane == 0) prev = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      prev = (unsigned int)__builtin_amdgcn_readfirstlane((int)prev);
      store = prev == (unsigned int)(lb - fb);
      if (store) {
        for (int b = fb; b <= lb; ++b) {
          const float* const src = part(b);
          v4f tmp[TMX];
#pragma unroll
          for (int t = 0; t < TMX; ++t) load_x4_agent(tmp[t], src + t * 256, lane_off);
#pragma unroll
          for (int t = 0; t < TMX; ++t) asm volatile("s_waitcnt vmcnt(0)" : "+v"(tmp[t]) : : "memory");
#pragma unroll
          for (int t = 0; t < TMX; ++t) {
            if (b == fb) acc[t] = tmp[t];
            else acc[t] += tmp[t];
          }
        }
        if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
      }
    }
    if (store) {
      const int m0 = at.begin + at.tile * C::kRows;
      const int n = at.chunk * kItemCols + wave * 16 + lg * 4;
      const int ring = (at.serial & (kRing - 1)) * 64;
#pragma unroll
      for (int t = 0; t < TMX; ++t) {
        const int r = t * 16 + l16;
        int m = m0 + r;
        if (m < at.end) {
          v4f v = acc[t];
          if (a.row_weight != nullptr) {
            const float rw = ring_weight[ring + r];
            v[0] *= rw; v[1] *= rw; v[2] *= rw; v[3] *= rw;
          }
          if (a.c_rows > 0) {
            m = ring_index[ring + r];
            if ((unsigned int)m >= (unsigned int)a.c_rows) continue;
          }
          store_output4<kModeBlock>(g, m, n, v);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < TMX; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    next_item(at);
    first_pair = 0;
  }
}

constexpr size_t part_bytes(int tmx) { return (size_t)kWaves * tmx * 256 * 4; }

template <int TMX>
int launch_stream_tmx(const StreamArgs& a, int grid, hipStream_t stream) {
  static PerDeviceFlags raised;
  void (*const kern)(StreamArgs) = fp8_gemm_stream_kernel<TMX>;
  const hipError_t e = raise_dynamic_lds_limit(raised, Cfg<TMX>::kLds, reinterpret_cast<const void*>(kern));
  if (e != hipSuccess) FG_FAIL(FG_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", Cfg<TMX>::kLds, hipGetErrorString(e));
  FG_LAUNCH(kern, dim3((uint32_t)grid), dim3(kThreads), Cfg<TMX>::kLds, stream, a);
  FG_CHECK_LAUNCH("fp8_gemm_stream_kernel");
  return FG_OK;
}

}  // namespace

int grouped_stream_rows(const GemmArgs& g, const GroupedGemm& gr) {
  const int64_t E = gr.n_groups;
  if (E < 1 || E > kMaxGroups || g.KB < 1) return 0;
  const int64_t scale_rows = (gr.row_index != nullptr && gr.index_div > 0) ? gr.x_rows : (int64_t)g.M;
  if (g.xs_cs < 0 || g.xs_rs < 0 || g.ws_cs < 0 || g.ws_rs < 0 || g.ws_cs >= (1 << 28) ||
      scale_rows * g.xs_rs + g.xs_cs >= (1ll << 29)) return 0;
  // steps are counted in 32 bits
  const int64_t chunks = ceil_div(g.N, (int64_t)kItemCols), pairs = (g.KB + 1) / 2;
  if ((g.M / 16 + E) * chunks * pairs >= (1ll << 30)) return 0;
  return grouped_stream_pass_rows(g.M, g.N, g.KB, E, cu_count());
}

int launch_grouped_stream(const GemmArgs& g, const GroupedGemm& gr, int rows, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  StreamArgs a = {};
  a.g = g;
  a.ends = gr.ends; a.n_groups = (int)gr.n_groups;
  a.w_group_stride = gr.w_group_stride; a.ws_group_stride = gr.ws_group_stride;
  a.row_index = gr.row_index; a.index_div = (int)gr.index_div; a.x_rows = (int)gr.x_rows;
  a.c_rows = (int)gr.c_rows; a.row_weight = gr.row_weight;
  a.chunks = (int)ceil_div(g.N, (int64_t)kItemCols);
  a.pairs = (g.KB + 1) / 2;
  a.min_steps = 4;
  const int tmx = rows / 16;
  int grid = cu_count();
  if (grid > 256) grid = 256;
  if (workspace != nullptr && (uintptr_t)workspace % 16 == 0 &&
      workspace_bytes >= FG_WORKSPACE_COUNTER_BYTES + (size_t)2 * grid * part_bytes(tmx)) {
    a.counters = reinterpret_cast<unsigned int*>(workspace);
    a.partials = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(workspace) + FG_WORKSPACE_COUNTER_BYTES);
  }
  if (tmx == 1) return launch_stream_tmx<1>(a, grid, stream);
  if (tmx == 2) return launch_stream_tmx<2>(a, grid, stream);
  return launch_stream_tmx<4>(a, grid, stream);
}

}  // namespace fg
