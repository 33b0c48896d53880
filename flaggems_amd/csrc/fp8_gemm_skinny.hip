// FP8 GEMM for few activation rows, or few tiles, on gfx950: tiles of 16 ... 128 rows x 32, 64 or 128 weight rows, both operands
// through LDS in a ring of deep stages; up to 128 rows one row of tiles, beyond that as many tiles as fill the chip once.
//
// What bounds it: the weight stream out of HBM.  A compute unit gets about 85 GB/s out of its L2 and 49 GB/s when the lines
// come from HBM, whatever is in flight beyond 40 KB, so the weights have to be spread over all units and the activations
// that every unit fetches again have to stay few: with 64 x 128 tiles they are half as many bytes as the weights.  Copies to
// LDS take whole lines (the fragment layout of the matrix instructions, 16 rows x 64 bytes a load, reaches a third of that).
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

// LDS of a block: a compute unit's for eight wavefronts, half of it for four
constexpr int skinny_table_bytes(int ring, int waves) {
  const int room = (waves == 8 ? 160 : 80) * 1024 - ring;
  return room < 24 * 1024 ? room : 24 * 1024;
}
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

// The instantiations, and their measured time in us (4700 problems of 1 to 128 rows, block scales and row / column scales, every
// split: the choice it leads to is 1-3 % slower than the fastest of all on average):
//   start + fullest * stages * (stage + rows * rows share) + bytes / stream + (rounds - 1) * round + (split ? exchange + fullest * part : 0)
// with `fullest` the blocks that the fullest compute unit works through.  Four wavefronts: two blocks on a unit.
struct SkinnyShape {
  int bm, bn, nst, waves;
  float start, stage, rows, stream_mb, round, exchange, part;
};
constexpr SkinnyShape kShapes[] = {
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
constexpr int kFirstOfRows = 6;
constexpr SkinnyShape kShapesOfRows[] = {
    {64, 32, 3, 4, 4.07f, 0.18f, 0.06f, 7.92f, 1.84f, 1.82f, 0.08f},
    {64, 64, 4, 8, 4.01f, 0.32f, 0.17f, 17.1f, 2.51f, 1.30f, 1.03f},
    {64, 128, 3, 8, 4.89f, 0.41f, 0.29f, 16.0f, 3.65f, 2.76f, 1.21f},
    {128, 64, 3, 8, 5.23f, 0.39f, 0.28f, 23.3f, 3.66f, 2.10f, 1.66f},
};

float skinny_cost(const SkinnyShape& sh, int64_t M, int64_t N, int64_t K, int64_t tiles, int64_t per, int64_t splits, int cus) {
  const int64_t blocks = tiles * splits, places = (int64_t)cus * (sh.waves == 4 ? 2 : 1), rounds = ceil_div(blocks, places);
  const float fullest = sh.waves == 4 ? (blocks <= cus ? 1.f : 2.f * (float)rounds) : (float)rounds;
  const float rows = (float)(ceil_div(M, 4) * 4 < sh.bm ? ceil_div(M, 4) * 4 : sh.bm) / (float)sh.bm;
  return sh.start + fullest * (float)per * (sh.stage + rows * sh.rows) + (float)N * (float)K * 1e-6f / sh.stream_mb + (float)(rounds - 1) * sh.round +
         (splits > 1 ? sh.exchange + fullest * sh.part : 0.f);
}

// Whether a block's scales fit beside its ring.
bool skinny_table_fits(const SkinnyShape& sh, int64_t stages) {
  const int64_t kbs = 2 * stages, room = skinny_table_bytes(sh.nst * (sh.bm + sh.bn) * 256, sh.waves);
  return (ceil_div((kbs | 1) * sh.bm, 64) * 64 + ceil_div(kbs, 64) * 64) * 4 <= room;
}

}  // namespace

// Where this kernel is the faster one (us, the kernels of the other files -> this one, both with their best split; M rows, N x K):
//  * up to 64 rows, K of 512 to 896: always (28, 4096 x 896: 5.6 -> 4.2; 16, 11584 x 896: 6.0 -> 4.5).
//  * up to 16 rows, K from 1024: unsplit in one round that fills over three quarters of the units; emptier rounds lose (12, 9216 x 5120:
//    12.0 -> 13.2).  Where the weight's rows lie 4 or 8 KB apart the other kernels' blocks meet on few memory channels: 24.9 -> 22.3 (1,
//    28672 x 4096), 27.8 -> 22.8 (16), 16.2 -> 13.6 (1, 8192 x 8192), 15.5 -> 12.7 (16, 14336 x 4096).  Otherwise from 9 rows, with the K that geometric
//    means of 60 to 160 problems a cell allow: 32-row tiles, block scales, K to 6144 0.92-0.98 (row and column scales 0.97-1.02); 64-row tiles,
//    block scales 0.87-0.96, row and column scales to 6144 0.93-0.99, past it 1.00-1.04; 128-row tiles, block scales 4096 to 8192 0.85-0.91 (2048
//    to 4096 1.02-1.04), row and column scales 0.89-1.01 (2048 to 4096 and past 8192 1.00-1.06).
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
//    8192 rows with K past 6144 do better on 128 x 128 tiles (128, 28672 x 4096: 34.8 -> 34.9; 104, 9664 x 13440 +23 %), and so do weights that one
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
SkinnyPlan plan_skinny(int64_t M, int64_t N, int64_t K, bool block_scales) {
  SkinnyPlan p = {};
  if (M < 1 || M > 4096 || N < (M > 1000 ? 128 : 512) || K < 512 || K % 128 != 0) return p;
  const int cus = cu_count();
  const int64_t stages = (K / 128 + 1) / 2, bytes = N * K, mb = 1000000;
  int best = -1;
  int64_t best_per = 0;
  const bool narrow_long = block_scales && M > 8 && M <= 16 && ((N <= (M > 12 ? 2560 : 1344) && K > 16384) || (N > 768 && N <= 1536 && K > 9216 && K <= 16384) ||
                                                                (N > 3584 && N <= 4096 && (K >= 14336 || (M > 12 && K > 10240))));
  if (M <= 16 && K >= 1024 && !narrow_long) {
    for (int c = 0; c < 3; ++c) {
      const int64_t tiles = ceil_div(N, (int64_t)kShapes[c].bn);
      if (tiles <= cus && tiles * 4 > (int64_t)cus * 3) best = c;
    }
    if (best < 0 || (block_scales && !skinny_table_fits(kShapes[best], stages))) return p;
    // (up to 8 rows with the shortest tiles only in a full round: 3, 6208 x 8192: 10.9 -> 12.1)
    const bool far_rows = K % 4096 == 0 && K <= 8192 && (best > 0 || M > 8 || ceil_div(N, (int64_t)kShapes[0].bn) * 16 > (int64_t)cus * 15);
    const bool use = best == 0 ? block_scales && K <= 6144 : best == 1 ? block_scales || K <= 6144 : K <= 8192 && (block_scales ? K >= 4096 : K < 2048 || K >= 4096);
    if (!far_rows && !(use && M > 8)) return p;
    best_per = stages;
  } else {
    bool use = (M <= 64 && K < 1024) || narrow_long;
    const int64_t units = ceil_div(M * N, (int64_t)8192);  // tiles of 128 x 64
    if (M <= 32) use = use || N > 6144 || (N > 4096 && (bytes <= 16 * mb || bytes >= 48 * mb)) || (N > 3072 && bytes >= 40 * mb) || (N >= 1024 && K >= 11008 && M * K >= 240000);
    else if (M <= 64) use = use || N >= 4096 || (N > 3072 && bytes >= 8 * mb) || (N >= 2048 && bytes >= 20 * mb) || (N >= 1536 && K >= 11008);
    else if (M <= 128) use = N <= 16384 && (N >= 8192 ? K <= 6144 : N > 4096 ? K >= 1024 : N >= 3072 ? K >= 3072 : (N >= 2048 && K >= 6144));
    else if (M <= 1000) use = units <= cus && (K <= 5120 || units <= 40 || (units <= 80 && K <= 8192) || (M <= 512 && K <= (block_scales ? 7168 : 8192) && units > 160)) &&
                              !(M <= 256 && N <= 1024 && bytes <= (N <= 768 ? 6 : 2) * mb) && !(M <= 512 && N <= 512 && bytes <= 2 * mb);
    else use = units <= cus && (M <= 2048 ? K <= 3072 || (K <= 4608 && N <= 768) : K <= 2560);
    if (!use) return p;
    const int first = M <= 16 ? 0 : M <= 32 ? 3 : M <= 64 ? 6 : M <= 128 ? 9 : kFirstOfRows, last = M <= 64 ? first + 3 : 10;
    float best_cost = 0.f, any_cost = 0.f;
    bool any_fits = true, one_round = true;
    for (int c = first; c < last; ++c) {
      const SkinnyShape& sh = M > 128 ? kShapesOfRows[c - kFirstOfRows] : kShapes[c];
      const int64_t tiles = ceil_div(N, (int64_t)sh.bn) * ceil_div(M, (int64_t)sh.bm);
      int64_t seen = 0;
      for (int64_t s = 1; s <= 12 && (s == 1 || tiles * s * 2 <= (int64_t)cus * 9); ++s) {
        const int64_t per = ceil_div(stages, s), splits = ceil_div(stages, per);
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
  const SkinnyShape& sh = kShapes[best];
  p.cfg = best;
  p.tiles_n = (int)ceil_div(N, (int64_t)sh.bn);
  p.tiles_m = (int)ceil_div(M, (int64_t)sh.bm);
  p.stages_per_split = (int)best_per;
  p.splits = (int)ceil_div(stages, best_per);
  const int64_t items = (int64_t)sh.bm * sh.bn / 256 / (sh.waves / 2), own = items > 1 ? items / 2 : 1;
  p.workspace_bytes = p.splits > 1 ? FG_WORKSPACE_COUNTER_BYTES + (size_t)p.tiles_n * p.tiles_m * p.splits * own * sh.waves * 64 * 16 : 0;
  p.use = true;
  return p;
}

// 32-bit offsets of a block's scales (strides are the caller's)
bool skinny_takes_scales(const GemmArgs& g, const SkinnyPlan& plan) {
  const int64_t kbs = 2 * (int64_t)plan.stages_per_split;
  return g.xs_rs >= 0 && g.xs_cs >= 0 && g.ws_cs >= 0 && g.xs_rs < (1 << 21) && g.xs_cs < (1 << 28) / kbs && g.ws_cs < (1 << 28) / kbs;
}

int launch_skinny(const GemmArgs& g, int mode, const SkinnyPlan& plan, void* workspace, hipStream_t stream) {
  const SkinnyShape& sh = kShapes[plan.cfg];
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
