// FP8 GEMM for few activation rows, or few tiles, on gfx950: tiles of 16 ... 128 rows x 32, 64 or 128 weight rows, both operands
// through LDS in a ring of deep stages; up to 128 rows one row of tiles, beyond that as many tiles as fill the chip once.
//
// What bounds it: the copies to LDS.  Alone, in this kernel's tiles, ring and order, a compute unit gets
//    119 GB/s (50 B/clk)  all 256 units the same lines, which their L2s hold
//     92                  216 tiles of 64 x 128 in six rows of tiles (333 rows, 4608 x 7168), weights left in the caches by the launch before
//     58                  the same with the weights out of HBM, 1.4 TB/s of them (23.8 us of the product's 26); 61 for 128 x 64 in two rows
//                         (256 rows, 8192 x 8192, 2.6 TB/s: 25.8 us)
//     35                  no tile shares its weights: 256 units take 6 TB/s, which is HBM's rate
// whatever is in flight beyond 40 KB.  So the weights have to be spread over all units, and the activations that every unit
// fetches again have to stay few: with 64 x 128 tiles they are half as many bytes as the weights.  The copies take whole lines (the
// fragment layout of the matrix instructions, 16 rows x 64 bytes a load, reaches a third of that).
//
//  * A stage is 256 bytes of K (two K-blocks) of every row: four rows an instruction, each 256 bytes in a run.  The
//    wavefronts form two groups; group g multiplies K-block 2 s + g of stage s.  One barrier per stage, that is per two
//    K-blocks.  The two groups' sums are added through LDS at the end, each group finishing half of the results.
//  * Blocks start at different stages of their K range and wrap round (`first stage` below).  All blocks in step read 256
//    bytes of every row at the same distance from the row's start; with rows a multiple of 4 KB apart those lie on few
//    memory channels.  Copies alone, N x K, rows in step -> rotated: 7168 x 16384 26.4 -> 21.5 us; 28672 x 4096 24.9 -> 20.8;
//    8192 x 8192 19.0 -> 12.4.
//  * Tiles of 32 weight rows (and some of 64) are a block of four wavefronts in half of LDS, two to a compute unit: one block's waits
//    are the other's work, and a tile count between one and two rounds leaves no unit empty.
//  * The scales of the block's K range come in before the first stage.
//  * K is split over blocks where the tiles do not fill the compute units; the wavefront that arrives last adds the
//    splits' sums in split order, so results do not depend on timing.
//
// Arithmetic as in the other kernels: per K-block products accumulated by the fp8 MFMA, multiplied by
// As[m, kb] * Bs[n / 128, kb] in fp32 (block mode) or accumulated unscaled and scaled at the end (row/column modes).

#include "fp8_gemm_common.h"
#include "fp8_gemm_skinny_plan.h"

#include <type_traits>

namespace fg {
namespace {

struct SkinnyArgs {
  GemmArgs g;
  int tiles_n, tiles_m, splits;
  int stages_per_split;  // stages of 256 bytes of K per block
  int table_row;         // block mode: floats of a row of the scale table in LDS (odd), or 0: the table is [K-block][row]
  uint32_t table_row_magic;  // ceil(2^32 / table_row): quotients of entry numbers below 2^16 by multiplication
  int table_ws;          // block mode: where the weight block's scales begin in the table (a multiple of 64)
  float* partials;       // [tile][split][item][thread] x 4 floats
  unsigned int* counters;  // one per tile and wavefront
};

template <int BM, int BN, int WM, int WN, int NST>
struct SkinnyCfg {
  static constexpr int kGroupWaves = WM * WN, kWaves = 2 * kGroupWaves, kThreads = kWaves * 64;
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  static constexpr int kItems = TM * TN, kOwn = kItems > 1 ? kItems / 2 : 1;  // results (16 x 16) of a wavefront, and those it finishes
  static constexpr int kStageBytes = (BM + BN) * 256;
  static constexpr int kRingBytes = NST * kStageBytes;
  static constexpr int kLoadsW = BN / 4 / kWaves;
  static constexpr int kSlabsX = BM / 4, kLoadsX = (kSlabsX + kWaves - 1) / kWaves;
  static_assert(BN % (4 * kWaves) == 0 && (kSlabsX % kWaves == 0 || kSlabsX < kWaves), "slabs must split evenly");
  static_assert(kWaves % 4 == 0, "a lane's chunk is the same in all its slabs");
  static_assert(kLoadsX <= 4 && (NST - 2) * (kLoadsW + kLoadsX) <= 63, "counted waits");
  static_assert(kItems == 1 || kItems % 2 == 0, "two groups share the results");
  static_assert(kItems * 64 * 16 * kWaves / 2 <= kRingBytes, "the groups exchange their sums in the ring");
  // scales of a block's K range (activation rows and weight block)
  static constexpr int kTableBytes = skinny_table_bytes(kRingBytes, kWaves);
  static constexpr int kLdsBytes = kRingBytes + kTableBytes;
};

__device__ __forceinline__ void skinny_copy_16(uint32_t byte_off, const void* base, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\t"
               "s_nop 0\n\t"
               "global_load_lds_dwordx4 %0, %1"
               :
               : "v"(byte_off), "s"(base), "s"(lds_addr)
               : "memory", "m0");
}
__device__ __forceinline__ void skinny_copy_4(uint32_t byte_off, const void* base, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\t"
               "s_nop 0\n\t"
               "global_load_lds_dword %0, %1"
               :
               : "v"(byte_off), "s"(base), "s"(lds_addr)
               : "memory", "m0");
}

template <int BM, int BN, int WM, int WN, int NST, int MODE>
__global__ __launch_bounds__(2 * WM* WN * 64) void fp8_gemm_skinny_kernel(SkinnyArgs a) {
  using Cfg = SkinnyCfg<BM, BN, WM, WN, NST>;
  constexpr int TM = Cfg::TM, TN = Cfg::TN, NT = Cfg::kThreads, kWaves = Cfg::kWaves;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];  // ring of stages [weights][activations], then the scales
  const GemmArgs& g = a.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int group = wave / Cfg::kGroupWaves, gw = wave % Cfg::kGroupWaves;
  const int wm0 = (gw % WM) * (BM / WM), wn0 = (gw / WM) * (BN / WN);
  const int l16 = lane & 15, lg = lane >> 4;

  // blocks of a split tile next to each other; with several rows of tiles, those against the same weights on one XCD (ids congruent
  // mod 8), whose L2 then has the weights after the first of them
  int tile, split, tile_m = 0;
  if (a.tiles_m == 1) {
    tile = (int)blockIdx.x / a.splits;
    split = (int)blockIdx.x - tile * a.splits;
  } else {
    const int share = (int)gridDim.x >> 3, rem = (int)gridDim.x & 7, xcd = (int)blockIdx.x & 7;
    const int at = xcd * share + (xcd < rem ? xcd : rem) + ((int)blockIdx.x >> 3), column = at / a.tiles_m;
    tile_m = at - column * a.tiles_m;
    split = column / a.tiles_n;
    tile = column - split * a.tiles_n;
  }
  const int n0 = tile * BN, m0 = tile_m * BM, rows = g.M - m0 < BM ? g.M - m0 : BM;
  const int stages_all = (g.KB + 1) >> 1;
  const int s_begin = split * a.stages_per_split;
  const int stages = (stages_all - s_begin < a.stages_per_split) ? stages_all - s_begin : a.stages_per_split;  // >= 1
  const int kb0 = s_begin * 2;
  const int kbs = (g.KB - kb0 < 2 * stages) ? g.KB - kb0 : 2 * stages;  // 2 * stages, or one fewer at the end of an odd K
  const int half_stage = (kbs & 1) ? stages - 1 : -1;                   // the stage with one K-block only

  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  float* const table = reinterpret_cast<float*>(lds + Cfg::kRingBytes);  // As of the block's rows and K range, then Bs

  // ---- this lane's bytes in a slab of four rows x 256 bytes: row lane >> 4, physical 16-byte chunk lane & 15 holds logical
  // chunk (lane & 15) ^ (row & 15).  Rows past the edge re-read the last valid row (never stored).
  const int chunk = (lane & 15) ^ ((wave & 3) * 4 + (lane >> 4));
  uint32_t w_off[Cfg::kLoadsW], x_off[Cfg::kLoadsX];
#pragma unroll
  for (int j = 0; j < Cfg::kLoadsW; ++j) {
    const int r = (wave + j * kWaves) * 4 + (lane >> 4), rc = r < g.N - n0 ? r : g.N - n0 - 1;
    w_off[j] = (uint32_t)rc * (uint32_t)g.ldw + (uint32_t)(chunk * 16);
  }
#pragma unroll
  for (int j = 0; j < Cfg::kLoadsX; ++j) {
    const int r = (wave + j * kWaves) * 4 + (lane >> 4), rc = r < rows ? r : rows - 1;
    x_off[j] = (uint32_t)rc * (uint32_t)g.ldx + (uint32_t)(chunk * 16);
  }
  // slabs of activations this wavefront copies: those past the last row stay as they are (a result depends on its own row)
  const int slabs_x = (rows + 3) / 4;
  const int loads_x = slabs_x > wave ? (slabs_x - wave + kWaves - 1) / kWaves : 0;
  // a stage that ends after its first K-block re-reads that instead of the bytes past K
  const uint32_t back = (chunk & 8) ? 128u : 0u;
  const uint8_t* const w_base = uniform_ptr(g.W + (int64_t)n0 * g.ldw + (int64_t)kb0 * 128);
  const uint8_t* const x_base = uniform_ptr(g.X + (int64_t)m0 * g.ldx + (int64_t)kb0 * 128);
  auto issue_stage = [&](int s, int slot) __attribute__((always_inline)) {
    const uint32_t sub = s == half_stage ? back : 0u;
    const uint32_t dst = lds_base + (uint32_t)(slot * Cfg::kStageBytes);
    const uint8_t* const w = w_base + (int64_t)s * 256;
    const uint8_t* const x = x_base + (int64_t)s * 256;
#pragma unroll
    for (int j = 0; j < Cfg::kLoadsW; ++j) skinny_copy_16(w_off[j] - sub, w, dst + (uint32_t)((wave + j * kWaves) * 1024));
#pragma unroll
    for (int j = 0; j < Cfg::kLoadsX; ++j)
      if (j < loads_x) skinny_copy_16(x_off[j] - sub, x, dst + (uint32_t)(BN * 256 + (wave + j * kWaves) * 1024));
  };

  // ---- ring: NST - 1 stages on their way while one is multiplied
  int s_load = (int)__umulhi((uint32_t)tile * 0x9E3779B9u, (uint32_t)stages);  // first stage: see the top of the file
  int s_mul = s_load;
  issue_stage(s_load, 0);
  s_load = s_load + 1 == stages ? 0 : s_load + 1;

  // ---- scales: entry i of the table is (row, K-block) with the K-blocks next to each other where they are in memory
  // (rows an odd number of floats apart: 16 rows of a K-block lie in 16 banks), else with the rows next to each other
  const int t_row = a.table_row ? a.table_row : 1, t_kb = a.table_row ? 1 : BM;
  if (MODE == kModeBlock) {
    const float* const xs_base = uniform_ptr(g.xs + (int64_t)m0 * g.xs_rs + (int64_t)kb0 * g.xs_cs);
    const int entries = a.table_row ? a.table_row * BM : kbs * BM;
    for (int i0 = wave * 64; i0 < entries; i0 += NT) {
      const uint32_t i = (uint32_t)(i0 + lane);
      int row = a.table_row ? (int)__umulhi(i, a.table_row_magic) : (int)(i % BM);
      int kb = a.table_row ? (int)i - row * a.table_row : (int)(i / BM);
      row = row < rows ? row : rows - 1;
      kb = kb < kbs ? kb : kbs - 1;
      const uint32_t off = (uint32_t)(row * (int)g.xs_rs + kb * (int)g.xs_cs) * 4u;  // the host checks that this fits
      skinny_copy_4(off, xs_base, lds_base + (uint32_t)(Cfg::kRingBytes + i0 * 4));
    }
    const float* const ws_row = uniform_ptr(g.ws + (int64_t)(n0 >> 7) * g.ws_rs + (int64_t)kb0 * g.ws_cs);
    for (int i0 = wave * 64; i0 < kbs; i0 += NT) {
      const int kb = i0 + lane < kbs ? i0 + lane : kbs - 1;
      skinny_copy_4((uint32_t)(kb * (int)g.ws_cs) * 4u, ws_row, lds_base + (uint32_t)(Cfg::kRingBytes + (a.table_ws + i0) * 4));
    }
  }

#pragma unroll
  for (int d = 1; d < NST - 1; ++d) {
    if (d < stages) {
      issue_stage(s_load, d);
      s_load = s_load + 1 == stages ? 0 : s_load + 1;
    }
  }
  v4f acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // stages that may still be on their way: vmcnt retires in order, and a wavefront counts its own copies
  auto wait_stages = [&](auto pending) __attribute__((always_inline)) {
    constexpr int p = decltype(pending)::value, w = Cfg::kLoadsW;
    if (p == 0 || loads_x == 0) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(p * w) : "memory");
    else if (Cfg::kLoadsX == 1 || loads_x == 1) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(p * (w + 1)) : "memory");
    else if (Cfg::kLoadsX == 2 || loads_x == 2) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(p * (w + 2)) : "memory");
    else if (Cfg::kLoadsX == 3 || loads_x == 3) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(p * (w + 3)) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" : : "n"(p * (w + 4)) : "memory");
  };
  // fragment of 16 rows: lane = row l16 (row & 15 of every group of 16), logical chunks lg and lg + 4 of this group's K-block
  const int frag_lo = l16 * 256 + (((group * 8 + lg) ^ l16) << 4), frag_hi = frag_lo ^ 64;
  int slot = 0;
  for (int s = 0; s < stages; ++s) {
    const int rem = stages - 1 - s;
    if (rem >= NST - 2) wait_stages(std::integral_constant<int, NST - 2>());
    else if (NST > 5 && rem == 3) wait_stages(std::integral_constant<int, 3>());
    else if (NST > 4 && rem == 2) wait_stages(std::integral_constant<int, 2>());
    else if (NST > 3 && rem == 1) wait_stages(std::integral_constant<int, 1>());
    else wait_stages(std::integral_constant<int, 0>());
    // (a bare barrier: __syncthreads() carries a fence for which the compiler waits for every copy in flight)
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
    if (s + NST - 1 < stages) {
      issue_stage(s_load, slot == 0 ? NST - 1 : slot - 1);
      s_load = s_load + 1 == stages ? 0 : s_load + 1;
    }
    const int kb = 2 * s_mul + group;
    if (kb < kbs) {  // uniform over the wavefront; false in the second group of the stage that holds one K-block
      const uint8_t* const tw = lds + slot * Cfg::kStageBytes + wn0 * 256;
      const uint8_t* const tx = lds + slot * Cfg::kStageBytes + BN * 256 + wm0 * 256;
      auto fragment = [&](const uint8_t* base, int rg) __attribute__((always_inline)) {
        const u32x4 lo = *reinterpret_cast<const u32x4*>(base + rg * 4096 + frag_lo);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(base + rg * 4096 + frag_hi);
        v8i f;
        f[0] = (int)lo.x; f[1] = (int)lo.y; f[2] = (int)lo.z; f[3] = (int)lo.w;
        f[4] = (int)hi.x; f[5] = (int)hi.y; f[6] = (int)hi.z; f[7] = (int)hi.w;
        return f;
      };
      v8i xf[TM], wf[TN];
#pragma unroll
      for (int j = 0; j < TM; ++j) xf[j] = fragment(tx, j);
#pragma unroll
      for (int i = 0; i < TN; ++i) wf[i] = fragment(tw, i);
      if (MODE == kModeBlock) {
        float sc[TM];
        const float ws = table[a.table_ws + kb];
#pragma unroll
        for (int j = 0; j < TM; ++j) sc[j] = table[(wm0 + j * 16 + l16) * t_row + kb * t_kb] * ws;
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j) {
            const v4f p = mfma_fp8_16x16x128(wf[i], xf[j], v4f{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(p[e], sc[j], acc[i][j][e]);
          }
      } else {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j)
            acc[i][j] = MODE == kModeRowColI8 ? mfma_i8_16x16x128(wf[i], xf[j], acc[i][j]) : mfma_fp8_16x16x128(wf[i], xf[j], acc[i][j]);
      }
    }
    s_mul = s_mul + 1 == stages ? 0 : s_mul + 1;
    slot = slot + 1 == NST ? 0 : slot + 1;
  }

  // ---- add the two groups: wavefront gw of group 0 and of group 1 hold the same results; group 0 finishes the first half of them,
  // group 1 the second (a lone result: group 0)
  auto add = [&](v4f x, v4f y) __attribute__((always_inline)) {
    if (MODE == kModeRowColI8) return __builtin_bit_cast(v4f, __builtin_bit_cast(v4i, x) + __builtin_bit_cast(v4i, y));
    return x + y;
  };
  constexpr int kItems = Cfg::kItems, kOwn = Cfg::kOwn;
  __syncthreads();  // the ring is read no more, and no copy is on its way
  v4f own[kOwn];
  {
    v4f* const area = reinterpret_cast<v4f*>(lds) + gw * kItems * 64 + lane;
#pragma unroll
    for (int t = 0; t < kItems; ++t) {
      const bool mine = kItems == 1 ? group == 0 : (t < kOwn) == (group == 0);
      if (!mine) area[t * 64] = acc[t / TM][t % TM];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kOwn; ++q) {
      if (kItems == 1) {
        own[0] = group == 0 ? add(acc[0][0], area[0]) : acc[0][0];
      } else if (group == 0) {
        own[q] = add(acc[q / TM][q % TM], area[q * 64]);
      } else {
        own[q] = add(area[(q + kOwn) * 64], acc[(q + kOwn) / TM][(q + kOwn) % TM]);
      }
    }
  }
  if (kItems == 1 && group != 0) return;

  // ---- K split over blocks: publish, count in, and let the wavefront that arrives last add the splits in order
  if (a.splits > 1) {
    const int id = tile * a.tiles_m + tile_m;
    const uint32_t t_off = (uint32_t)tid * 16u;
    constexpr int kSlotFloats = kOwn * NT * 4;
    float* const slots = uniform_ptr(a.partials + (size_t)id * a.splits * kSlotFloats);
    {
      float* const mine = uniform_ptr(slots + (size_t)split * kSlotFloats);
#pragma unroll
      for (int q = 0; q < kOwn; ++q) store_x4_agent(mine + q * NT * 4, t_off, own[q]);
    }
    wait_vmem_all();
    unsigned int* const cnt = a.counters + id * kWaves + wave;
    unsigned int prev = 0;
    if (lane == 0) prev = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    prev = (unsigned int)__builtin_amdgcn_readfirstlane((int)prev);
    if (prev != (unsigned int)(a.splits - 1)) return;
    // four splits' sums on their way at a time (a round trip to memory each time), added in split order
    constexpr int kBatch = 4;
    for (int s0 = 0; s0 < a.splits; s0 += kBatch) {
      v4f tmp[kBatch][kOwn];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int s = s0 + b < a.splits ? s0 + b : a.splits - 1;  // past the end: re-read the last split, unused
        const float* const src = uniform_ptr(slots + (size_t)s * kSlotFloats);
#pragma unroll
        for (int q = 0; q < kOwn; ++q) load_x4_agent(tmp[b][q], src + q * NT * 4, t_off);
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b)  // the values are operands of the wait, so no use can move above it
#pragma unroll
        for (int q = 0; q < kOwn; ++q) asm volatile("s_waitcnt vmcnt(0)" : "+v"(tmp[b][q]) : : "memory");
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        if (s0 + b < a.splits) {
#pragma unroll
          for (int q = 0; q < kOwn; ++q) own[q] = s0 + b == 0 ? tmp[b][q] : add(own[q], tmp[b][q]);  // (no "0 + x" in the sum)
        }
      }
    }
    if (lane == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
  }

  // ---- results: the lane holds m = m0 + wm0 + j * 16 + l16, n = n0 + wn0 + i * 16 + 4 * lg + [0, 4)
#pragma unroll
  for (int q = 0; q < kOwn; ++q) {
    const int t = kItems > 1 && group ? q + kOwn : q;
    const int i = t / TM, j = t % TM;
    const int m = m0 + wm0 + j * 16 + l16;
    if (m < g.M) store_output4<MODE>(g, m, n0 + wn0 + i * 16 + lg * 4, own[q]);
  }
}

template <int BM, int BN, int WM, int WN, int NST>
int launch_skinny_cfg(SkinnyArgs sa, const SkinnyPlan& plan, int mode, hipStream_t stream) {
  using Cfg = SkinnyCfg<BM, BN, WM, WN, NST>;
  auto kb = fp8_gemm_skinny_kernel<BM, BN, WM, WN, NST, kModeBlock>;
  auto kr = fp8_gemm_skinny_kernel<BM, BN, WM, WN, NST, kModeRowCol>;
  auto ki = fp8_gemm_skinny_kernel<BM, BN, WM, WN, NST, kModeRowColI8>;
  static PerDeviceFlags lds_limit_raised = {};  // per instantiation
  {
    const hipError_t e = raise_dynamic_lds_limit(lds_limit_raised, Cfg::kLdsBytes, reinterpret_cast<const void*>(kb),
                                                  reinterpret_cast<const void*>(kr), reinterpret_cast<const void*>(ki));
    if (e != hipSuccess) FG_FAIL(FG_ERR_LAUNCH, "hipFuncSetAttribute(%d bytes LDS): %s", Cfg::kLdsBytes, hipGetErrorString(e));
  }
  const dim3 grid((uint32_t)(sa.tiles_n * sa.tiles_m * sa.splits)), block(Cfg::kThreads);
  if (mode == kModeBlock) FG_LAUNCH(kb, grid, block, Cfg::kLdsBytes, stream, sa);
  else if (mode == kModeRowColI8) FG_LAUNCH(ki, grid, block, Cfg::kLdsBytes, stream, sa);
  else FG_LAUNCH(kr, grid, block, Cfg::kLdsBytes, stream, sa);
  FG_CHECK_LAUNCH("fp8_gemm_skinny_kernel");
  return FG_OK;
}

}  // namespace

// 32-bit offsets of a block's scales (strides are the caller's)
bool skinny_takes_scales(const GemmArgs& g, const SkinnyPlan& plan) {
  const int64_t kbs = 2 * (int64_t)plan.stages_per_split;
  return g.xs_rs >= 0 && g.xs_cs >= 0 && g.ws_cs >= 0 && g.xs_rs < (1 << 21) && g.xs_cs < (1 << 28) / kbs && g.ws_cs < (1 << 28) / kbs;
}

int launch_skinny(const GemmArgs& g, int mode, const SkinnyPlan& plan, void* workspace, hipStream_t stream) {
  const SkinnyShape& sh = kSkinnyShapes[plan.cfg];
  const int kbs = 2 * plan.stages_per_split;
  SkinnyArgs sa = {};
  sa.g = g;
  sa.tiles_n = plan.tiles_n;
  sa.tiles_m = plan.tiles_m;
  sa.splits = plan.splits;
  sa.stages_per_split = plan.stages_per_split;
  if (mode == kModeBlock) {
    sa.table_row = g.xs_cs == 1 ? kbs | 1 : 0;
    sa.table_row_magic = sa.table_row ? (uint32_t)ceil_div((int64_t)1 << 32, (int64_t)sa.table_row) : 0;
    sa.table_ws = (int)(ceil_div((int64_t)(sa.table_row ? sa.table_row : kbs) * sh.bm, (int64_t)64) * 64);
  }
  if (plan.splits > 1) {
    sa.counters = reinterpret_cast<unsigned int*>(workspace);
    sa.partials = reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + FG_WORKSPACE_COUNTER_BYTES);
  }
  switch (plan.cfg) {
    case 0: return launch_skinny_cfg<16, 32, 1, 2, 6>(sa, plan, mode, stream);
    case 1: return launch_skinny_cfg<16, 64, 1, 2, 3>(sa, plan, mode, stream);
    case 2: return launch_skinny_cfg<16, 128, 1, 4, 4>(sa, plan, mode, stream);
    case 3: return launch_skinny_cfg<32, 32, 1, 2, 4>(sa, plan, mode, stream);
    case 4: return launch_skinny_cfg<32, 64, 1, 2, 3>(sa, plan, mode, stream);
    case 5: return launch_skinny_cfg<32, 128, 1, 4, 3>(sa, plan, mode, stream);
    case 6: return launch_skinny_cfg<64, 32, 2, 1, 3>(sa, plan, mode, stream);
    case 7: return launch_skinny_cfg<64, 64, 2, 2, 4>(sa, plan, mode, stream);
    case 8: return launch_skinny_cfg<64, 128, 2, 2, 3>(sa, plan, mode, stream);
    default: return launch_skinny_cfg<128, 64, 2, 2, 3>(sa, plan, mode, stream);
  }
}

}  // namespace fg
