// Device code of the persistent kernel, whose wavefront groups alternate between fetching and multiplying
// (fp8_gemm_pingpong.hip): fragments in LDS, matrix instructions written out in assembly, and
// the stores of a wavefront's results.
#pragma once

#include "fp8_gemm_common.h"

namespace fg {
namespace {

constexpr int kTN = 8, kTM = 4;  // MFMA tiles of the persistent kernel's wavefronts: 128 weight rows x 64 activation rows

// weight row (within the wavefront's 128) held by LDS row rho of the wavefront's region
__device__ __forceinline__ int weight_row_of_lds_row(int rho) {
  const int t = rho >> 4, i = rho & 15;
  return (t >> 1) * 32 + (i >> 2) * 8 + (t & 1) * 4 + (i & 3);
}
// first of the eight consecutive output columns that lane group lg holds in MFMA tiles 2q and 2q+1
__device__ __forceinline__ int piece_column(int n_base, int q, int lg) { return n_base + q * 32 + lg * 8; }

__device__ __forceinline__ int fragment_offset(int lane) {
  const int r = lane & 15, g = lane >> 4;
  return r * 128 + ((g ^ (r & 7)) << 4);
}

__device__ __forceinline__ v8i read_frag(const uint8_t* region, int rg, int lane_off) {
  const u32x4 lo = *reinterpret_cast<const u32x4*>(region + rg * 2048 + lane_off);
  const u32x4 hi = *reinterpret_cast<const u32x4*>(region + rg * 2048 + (lane_off ^ 64));
  v8i f;
  f[0] = (int)lo.x; f[1] = (int)lo.y; f[2] = (int)lo.z; f[3] = (int)lo.w;
  f[4] = (int)hi.x; f[5] = (int)hi.y; f[6] = (int)hi.z; f[7] = (int)hi.w;
  return f;
}

// MFMA with a zero accumulator input, result in architectural VGPRs
__device__ __forceinline__ v4f mfma_partial(const v8i& w, const v8i& x) {
  v4f p = {};
  asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=&v"(p) : "v"(w), "v"(x));
  return p;
}

__device__ __forceinline__ void mfma_accumulate(v4f& c, const v8i& w, const v8i& x) {
  asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+v"(c) : "v"(w), "v"(x));
}

// int8 operands (kModeRowColI8): the same fragment as two 16x16x64 products (`half` = 0: the lane's first 16 bytes of
// the K-block, 1: its second 16), int32 sums kept as bit patterns in the accumulator registers; the two instructions
// take as long as the one fp8 instruction.  The multiply phase issues the two halves of one accumulator kTM
// instructions apart, so that the matrix pipe never waits for the sum it has just started.
// bf16 and fp16 operands (kModeRowColBF16 / F16) take the same route: a lane's 16 bytes are eight elements, the
// fragment two 16x16x32 products into fp32 sums, and the pair again takes as long as the one fp8 instruction.
template <int MODE>
__device__ __forceinline__ void mfma_accumulate_half(v4f& c, const v8i& w, const v8i& x, int half) {
  typedef int v4i_ __attribute__((ext_vector_type(4)));
  const v4i_ wh = half ? v4i_{w[4], w[5], w[6], w[7]} : v4i_{w[0], w[1], w[2], w[3]};
  const v4i_ xh = half ? v4i_{x[4], x[5], x[6], x[7]} : v4i_{x[0], x[1], x[2], x[3]};
  if constexpr (MODE == kModeRowColBF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(wh), "v"(xh));
  else if constexpr (MODE == kModeRowColF16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(wh), "v"(xh));
  else asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(c) : "v"(wh), "v"(xh));
}

// Scales that are powers of two (POW2): the block-scaled form of the instruction multiplies the products by
// 2^(sw - 127) * 2^(sx - 127) on their way into the sum, so the matrix pipe accumulates the scaled K-blocks itself and
// the multiply phase has no vector-ALU work at all.  sw / sx: E8M0 exponent in the low byte of a register per lane,
// taken for the operand row the lane holds (lane & 15); every 32-element K group of a row gets the same one here.
__device__ __forceinline__ void mfma_scaled_accumulate(v4f& c, const v8i& w, const v8i& x, int sw, int sx) {
  asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[0,0,0] op_sel_hi:[0,0,0]"
               : "+v"(c)
               : "v"(w), "v"(x), "v"(sw), "v"(sx));
}
__device__ __forceinline__ int e8m0_of(float s) { return (int)((float_to_bits(s) >> 23) & 0xFFu); }

// acc += p * s.  A wavefront issues one instruction every four cycles and the matrix pipe takes an MFMA of
// this shape every 32, so a multiply step has eight issue slots: the MFMA, these four FMAs and three spare
// (LDS reads, tile loads).  p is the result of the MFMA issued TWO steps earlier: at least 64 cycles have
// passed since its issue, more than the 11 wait states (44 cycles) gfx950 requires between an 8-pass MFMA
// write and a VALU read, so no s_nop is spent in the steady state.  NOPS > 0 pads the tail of the phase.
template <int NOPS>
__device__ __forceinline__ void scale_into(v4f& acc, const v4f& p, float s) {
  float a0 = acc[0], a1 = acc[1], a2 = acc[2], a3 = acc[3];
  if (NOPS > 0) {
    asm volatile("s_nop %9\n\t"
                 "v_fmac_f32 %0, %4, %8\n\t"
                 "v_fmac_f32 %1, %5, %8\n\t"
                 "v_fmac_f32 %2, %6, %8\n\t"
                 "v_fmac_f32 %3, %7, %8"
                 : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
                 : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(s), "n"(NOPS - 1));
  } else {
    asm volatile("v_fmac_f32 %0, %4, %8\n\t"
                 "v_fmac_f32 %1, %5, %8\n\t"
                 "v_fmac_f32 %2, %6, %8\n\t"
                 "v_fmac_f32 %3, %7, %8"
                 : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3)
                 : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(s));
  }
  acc[0] = a0; acc[1] = a1; acc[2] = a2; acc[3] = a3;
}

template <int PENDING>
__device__ __forceinline__ void wait_vmem() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(PENDING) : "memory");
}

// 16 bytes of results
__device__ __forceinline__ void store_result_16(uint16_t* p, u32x4 v) {
  *reinterpret_cast<u32x4*>(p) = v;
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const bf16x2_t h = __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t);
  return __builtin_bit_cast(uint32_t, h);
}
// Two results as the 16-bit output type, F16: fp16, else bf16 (round to nearest even both).  The empty statement
// keeps the compiler from folding a multiplication that produced the value into the conversion (one rounding
// instead of the two that the tile kernels and the reference perform).
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
template <bool F16>
__device__ __forceinline__ uint32_t pack_out(float lo, float hi) {
  if (!F16) return pack_bf16(lo, hi);
  asm volatile("" : "+v"(lo), "+v"(hi));
  const f16x2_t h = {(_Float16)lo, (_Float16)hi};
  return __builtin_bit_cast(uint32_t, h);
}
// the two halves of such a word as fp32
template <bool F16>
__device__ __forceinline__ float unpack_lo(uint32_t w) {
  return F16 ? (float)__builtin_bit_cast(f16x2_t, w)[0] : bits_to_float(w << 16);
}
template <bool F16>
__device__ __forceinline__ float unpack_hi(uint32_t w) {
  return F16 ? (float)__builtin_bit_cast(f16x2_t, w)[1] : bits_to_float(w & 0xFFFF0000u);
}

// The value that the lane holding the neighbouring row (l16 ^ 1, same lg: the adjacent lane) has in `v`.
__device__ __forceinline__ uint32_t from_row_neighbour(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1 /* quad_perm [1, 0, 3, 2] */, 0xF, 0xF, true);
}
// Two pieces that are neighbours in a row (64 + 64 bytes: `lo` the lower columns) leave as whole 128-byte runs: the
// lanes of an even row and of the odd row after it exchange one piece each, after which the eight lanes of such a pair
// of rows hold the 128 bytes of the even row (first store) and of the odd row (second store).  A store instruction
// then touches 8 memory lines instead of 16 halves, and the time a compute unit's address unit spends on a store
// goes with the lines it touches: measured on whole launches at M = 4096, N = 32768, K = 512: 103 -> 92 us;
// N = 24576, K = 1536: 160 -> 150 us; N = 7168, K = 2304: 74 -> 69 us.
// `even_row`: the lane's position in the even row of its pair, at the columns of `lo` (odd lanes: of `hi`).
__device__ __forceinline__ void store_piece_pair(uint16_t* even_row, int64_t ldc, bool odd, const uint32_t (&lo)[4], const uint32_t (&hi)[4]) {
  u32x4 first, second;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t lo_there = from_row_neighbour(lo[e]), hi_there = from_row_neighbour(hi[e]);
    first[e] = odd ? hi_there : lo[e];
    second[e] = odd ? hi[e] : lo_there;
  }
  store_result_16(even_row, first);
  store_result_16(even_row + ldc, second);
}

// Stores the wavefront's 64 x 128 results as bf16.  Lane (l16, lg) holds, for every activation tile j, four
// pieces of eight consecutive columns of row m_base + 16 j + l16: piece q starts at column
// n_base + 32 q + 8 lg and comes from MFMA tiles 2q and 2q+1.  The host guarantees ldc % 8 == 0 and a 16-byte
// aligned C, so a piece leaves as one 16-byte store, and the four lanes of a row cover 64 contiguous bytes per
// store instruction (tiles with edges), or pairs of pieces leave as whole 128-byte runs (ALIGNED: store_piece_pair).
// Row/column mode: the sums are scaled by a_scale[m] * b_scale[n] first, and the bias is added to the rounded
// value, in bf16, as the reference's epilogue does (src/flag_gems/fused/cutlass_scaled_mm.py:288-305).
// ALIGNED: the tile lies inside the matrix; a wavefront then issues exactly kStoresPerTile store instructions.
constexpr int kStoresPerTile = 16;
// SCATTER (grouped problems): rows go where out_index says (see PpArgs::c_rows).
// JN: activation fragments per wavefront (rows m_base .. m_base + 16 JN).
// F16: the results are fp16 (else bf16).
// NT, q0: `acc` holds the NT MFMA tiles of pieces q0 .. q0 + NT / 2 - 1 (all eight, or the half that the finish of a
// shared tile sums at a time).
template <int MODE, bool ALIGNED, bool SCATTER = false, int JN = kTM, bool F16 = false, int NT = kTN>
__device__ __forceinline__ void store_tile(const GemmArgs& a, const v4f (&acc)[NT][JN], int m_base, int n_base,
                                           int l16, int lg, int m_end, const int* out_index = nullptr, int c_rows = 0,
                                           const float* row_weight = nullptr, int q0 = 0) {
  if constexpr (!ALIGNED && !SCATTER && NT % 4 == 0 && MODE == kModeBlock) {
    // a wavefront's share that lies inside the matrix (uniform) takes the stores of whole tiles (block scales only:
    // the row/column modes' instantiations with edges have no registers left for a second store path and spill)
    if (m_base + 16 * JN <= m_end && piece_column(n_base, q0 + NT / 2, 0) <= a.N) {
      store_tile<MODE, true, false, JN, F16, NT>(a, acc, m_base, n_base, l16, lg, m_end, nullptr, 0, nullptr, q0);
      return;
    }
  }
  constexpr bool kPairs = ALIGNED && !SCATTER && NT % 4 == 0;  // whole tiles: pieces leave two at a time
  const bool odd = (l16 & 1) != 0;
  if (MODE != kModeBlock) {
    uint32_t kept[JN][4];  // kPairs: the lower piece of the pair, while the upper one is computed
    (void)kept;
    // eight columns at a time, so that only eight column scales and bias values are live
#pragma unroll
    for (int q = 0; q < NT / 2; ++q) {
      const int n = piece_column(n_base, q0 + q, lg);
      const bool full = ALIGNED || n + 8 <= a.N;
      float sb[8], bias[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int ne = n + e < a.N ? n + e : a.N - 1;
        sb[e] = a.ws[a.ws_per_col ? ne : 0];
        bias[e] = a.bias ? load_as_float(a.bias, ne, a.bias_dtype) : 0.f;
      }
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        const int m = m_base + j * 16 + l16;
        if (!ALIGNED && m >= m_end) continue;
        const float sa = a.xs[a.xs_per_row ? m : 0];
        uint32_t w[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {  // two columns per word
          const int t = 2 * q + (h >> 1), e0 = (h & 1) * 2;
          // (int8 operands: the registers hold int32 sums.  The element is copied to a scalar before the bit cast:
          // a bit cast applied to the vector element itself reads element 0 whatever the index.)
          const float r0 = acc[t][j][e0], r1 = acc[t][j][e0 + 1];
          const float s0 = MODE == kModeRowColI8 ? (float)__float_as_int(r0) : r0;
          const float s1 = MODE == kModeRowColI8 ? (float)__float_as_int(r1) : r1;
          float v0 = (s0 * sa) * sb[4 * (h >> 1) + e0];
          float v1 = (s1 * sa) * sb[4 * (h >> 1) + e0 + 1];
          if (MODE >= kModeRowColBF16) {  // one rounding, the bias before it
            if (a.bias) { v0 = v0 + bias[4 * (h >> 1) + e0]; v1 = v1 + bias[4 * (h >> 1) + e0 + 1]; }
            w[h] = pack_out<F16>(v0, v1);
            continue;
          }
          w[h] = pack_out<F16>(v0, v1);
          if (a.bias)
            w[h] = pack_out<F16>(unpack_lo<F16>(w[h]) + bias[4 * (h >> 1) + e0],
                                 unpack_hi<F16>(w[h]) + bias[4 * (h >> 1) + e0 + 1]);
        }
        if constexpr (kPairs) {
          if ((q & 1) == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) kept[j][e] = w[e];
          } else {
            // (q0 + q is odd: this lane's columns of the lower piece start 32 columns before n)
            store_piece_pair(reinterpret_cast<uint16_t*>(a.C) + (int64_t)(m - (l16 & 1)) * a.ldc + n - 32 + (l16 & 1) * 32,
                             a.ldc, odd, kept[j], w);
          }
          continue;
        }
        uint16_t* const cp = reinterpret_cast<uint16_t*>(a.C) + (int64_t)m * a.ldc + n;
        if (full) {
          *reinterpret_cast<u32x4*>(cp) = u32x4{w[0], w[1], w[2], w[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < a.N) cp[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
        }
      }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < JN; ++j) {
    const int m = m_base + j * 16 + l16;
    if (!ALIGNED && m >= m_end) continue;
    int64_t out_row = m;
    float wgt = 1.f;
    if (SCATTER && out_index != nullptr) {
      const int idx = out_index[m];
      if (idx < 0 || idx >= c_rows) continue;
      out_row = idx;
      if (row_weight != nullptr) wgt = row_weight[idx];
    }
    uint16_t* const row = reinterpret_cast<uint16_t*>(a.C) + out_row * a.ldc;
    uint32_t w[2 * NT];
    if (SCATTER && row_weight != nullptr) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        w[2 * t] = pack_out<F16>(acc[t][j][0] * wgt, acc[t][j][1] * wgt);
        w[2 * t + 1] = pack_out<F16>(acc[t][j][2] * wgt, acc[t][j][3] * wgt);
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        w[2 * t] = pack_out<F16>(acc[t][j][0], acc[t][j][1]);
        w[2 * t + 1] = pack_out<F16>(acc[t][j][2], acc[t][j][3]);
      }
    }
    if constexpr (kPairs) {
#pragma unroll
      for (int q = 0; q < NT / 2; q += 2) {
        const uint32_t lo[4] = {w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]};
        const uint32_t hi[4] = {w[4 * q + 4], w[4 * q + 5], w[4 * q + 6], w[4 * q + 7]};
        store_piece_pair(reinterpret_cast<uint16_t*>(a.C) + (int64_t)(m - (l16 & 1)) * a.ldc + piece_column(n_base, q0 + q, lg) + (l16 & 1) * 32,
                         a.ldc, odd, lo, hi);
      }
      continue;
    }
#pragma unroll
    for (int q = 0; q < NT / 2; ++q) {
      const int n = piece_column(n_base, q0 + q, lg);
      if (ALIGNED || n + 8 <= a.N) {
        store_result_16(row + n, u32x4{w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]});
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (n + e < a.N) row[n + e] = (uint16_t)(w[4 * q + (e >> 1)] >> (16 * (e & 1)));
      }
    }
  }
}

}  // namespace
}  // namespace fg
