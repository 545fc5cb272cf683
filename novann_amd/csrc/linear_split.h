// Linear products of any shape on bf16 MFMA with K split over the waves of a
// workgroup (gfx950), for the shapes the whole-tile kernels do not take or
// would leave most of the chip idle on: few rows, ragged sides, and the
// backward's products on operands that lie K-major.
//
//   y[m, n] = epilogue(s * sum over k of X(m, k) * W(n, k))
//
// A workgroup owns one small tile (16 MT x 16 NT outputs) and its NWV waves
// take contiguous runs of 64-K blocks of it, each wave with the whole tile's
// accumulators: v_mfma_f32_16x16x32_bf16 with W as the A operand, so a lane
// ends with 4 consecutive n of one m.  Operands go from global memory straight
// into fragment registers -- a K slice is read by exactly one wave, so LDS
// staging would share nothing -- with no barrier until the K loop ends; the
// waves' partial tiles are then added in wave order through LDS (a fixed
// order: results are reproducible), 16 rows at a time, and stored with the
// epilogue in 4-element runs along n.
//
// Each operand comes in one of two layouts:
//   row: K contiguous (long products: LsQuad instead).  In block k0, lane (r, g)
//        (r = lane % 16, g = lane / 16) loads the 16 consecutive elements
//        k0 + 16 g .. + 15 of row 16 t + r for tile t: two MFMA steps of 8.
//   col: K-major (element (k, m) at k * pitch + m).  The lane loads, for each
//        of the same 16 k, the T consecutive elements T r .. T r + T - 1 (T
//        tiles): element t of every run makes tile t's fragment, so tile t
//        holds the indices T r + t and no lane exchange is needed (M or N at
//        least T).
// Both orders of K agree, which is all a product needs.  Rows need not start
// on any boundary beyond their element (gfx950 loads vectors at any address);
// the last block, when K % 64 != 0, is loaded element by element with zeros
// past K, and indices past M or N are clamped to the last one (never stored).
//
// What bounds it: a CU's load rate times the operand bytes of a tile, then
// latency; so the tile is 64 x 64 (4 waves, two workgroups a CU) when those
// tiles cover the CUs, 32 x 32 on 8 waves below that, and 16 x 16 on 16 waves
// for at most 16 rows (every CU then streams its own 16 rows of W).  A fragment
// load straight from 16 rows reaches a line a lane and the CU only 94 GB/s of
// them, whatever the depth of the pipeline (2 to 8 half blocks in flight: the
// same time); row operands of long products are therefore read as LsQuad says.
// Measured (E4M3 W 4096 x 4096, fp32 x, warm MALL; the guarded 128 x 256-tile
// kernel it replaced in brackets): 1 row 6.8 us (296), 16 rows 8.4 (306), 64
// rows 15.7 (342), 14.6 with FP4 W, 9.6 with bf16 x too; 500 x 1024 x 1024 12.6
// (120); 333 x 777 x 1111 16.8 (277).  Large products that the tile kernels' ragged
// forms cannot read run here too: fp32 W 2048 x 4096 x 4096 458 (672), E4M3 W 2000
// x 4095 x 4096 476 (1339), FP4 W 2048 x 4080 x 4096 277 (868), E4M3 x and W 2000
// x 4096 x 4096 124 (355).  (The 1 row kernel is 7.4 to 7.6 us in a kernel trace,
// which adds to short ones; 6.8 between events over a run of launches.)
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "novaq_convert.h"
#include "novaq_epilogue.h"
#include "novaq_internal.h"
#include "novaq_split_index.h"
#include "novaq_xload.h"

namespace novaq {
namespace {

typedef __bf16 ls_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ls_f32x4 __attribute__((ext_vector_type(4)));
// vectors at any byte address
typedef uint32_t ls_u32x4u __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t ls_u32x2u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t ls_u32u __attribute__((aligned(1)));
typedef uint16_t ls_u16u __attribute__((aligned(1)));

constexpr int LS_KB = 64;  // K per block: 16 elements a lane

__device__ __forceinline__ uint32_t ls_pair(float a, float b) {
  const xl_f32x2 f = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, xl_bf16x2));
}

// Two f16 values of a word as two bf16 (through the exact fp32 widening).
__device__ __forceinline__ uint32_t ls_f16_pair(uint32_t word) {
  const xl_f32x2 f = __builtin_convertvector(__builtin_bit_cast(xl_f16x2, word), xl_f32x2);
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, xl_bf16x2));
}

// Code of element e of a row in storage order.
template <int DT>
__device__ __forceinline__ uint32_t ls_code(const uint8_t* row, int64_t e) {
  if constexpr (dtype_bits(DT) == 32) return *reinterpret_cast<const ls_u32u*>(row + 4 * e);
  else if constexpr (dtype_bits(DT) == 16) return *reinterpret_cast<const ls_u16u*>(row + 2 * e);
  else if constexpr (dtype_bits(DT) == 8) return row[e];
  else return (row[e >> 1] >> ((e & 1) * 4)) & 0xFu;
}

// 8 consecutive stored elements (words w[0 ..]) as bf16.
template <int DT>
__device__ __forceinline__ ls_bf16x8 ls_decode8(const uint32_t* w) {
  uint32_t o[4];
  if constexpr (DT == F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = ls_pair(u2f(w[2 * i]), u2f(w[2 * i + 1]));
  } else if constexpr (DT == BF16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = w[i];
  } else if constexpr (DT == F16) {
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = ls_f16_pair(w[i]);
  } else if constexpr (DT == E2M1) {
    const uint32_t v = w[0];
    o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, 1.0f, 0));
    o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, 1.0f, 1));
    o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, 1.0f, 2));
    o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(v, 1.0f, 3));
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t v = w[i];
      if constexpr (DT == E4M3) {
        o[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, false));
        o[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, true));
      } else {
        o[2 * i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(v, 1.0f, false));
        o[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(v, 1.0f, true));
      }
    }
  }
  return __builtin_bit_cast(ls_bf16x8, make_uint4(o[0], o[1], o[2], o[3]));
}

// Row operand: T tiles of 16 rows, K contiguous.  Wide elements are loaded a
// half block (8 a lane, one MFMA step) at a time, 8- and 4-bit codes a whole
// block at a time (16- and 8-byte loads).
template <int DT, int T>
struct LsRow {
  static constexpr int bits = dtype_bits(DT);
  static constexpr bool HALF = bits >= 16;
  static constexpr int NE = HALF ? 8 : 16;        // elements a load takes
  static constexpr int NW = NE * bits / 32;       // words of them
  typedef uint32_t Run __attribute__((ext_vector_type(NW)));
  struct Regs {
    Run w[T];
  };
  const uint8_t* row[T];
  int kl;  // the lane's first element within a block

  __device__ __forceinline__ void init(const uint8_t* p, int64_t pitch, int i0, int count, int lane) {
    kl = (lane >> 4) * 16;
#pragma unroll
    for (int t = 0; t < T; ++t) row[t] = p + (int64_t)min(i0 + 16 * t + (lane & 15), count - 1) * pitch;
  }
  // elements k0 + kl + 8 u ..
  __device__ __forceinline__ void load(Regs& r, int k0, const int u) const {
    const int64_t b = (int64_t)(k0 + kl + 8 * u) * bits / 8;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const uint8_t* p = row[t] + b;
      if constexpr (NW == 8) {
        const ls_u32x4u lo = *reinterpret_cast<const ls_u32x4u*>(p);
        const ls_u32x4u hi = *reinterpret_cast<const ls_u32x4u*>(p + 16);
        r.w[t] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      } else {
        typedef Run RunU __attribute__((aligned(1)));
        r.w[t] = *reinterpret_cast<const RunU*>(p);
      }
    }
  }
  __device__ __forceinline__ void load_tail(Regs& r, int k0, const int u, int K) const {
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        uint32_t v = 0;
#pragma unroll
        for (int e = 0; e < 32 / bits; ++e) {
          const int k = k0 + kl + 8 * u + i * (32 / bits) + e;
          if (k < K) v |= ls_code<DT>(row[t], k) << ((e * bits) & 31);
        }
        r.w[t][i] = v;
      }
    }
  }
  // load_tail for K >= NE (even for 4-bit codes) with few instructions: a run
  // that would pass K is read ending at K and shifted down to its place, zeros
  // behind it.
  __device__ __forceinline__ void load_end(Regs& r, int k0, const int u, int K) const {
    const int k = k0 + kl + 8 * u;
    const int from = min(k, K - NE), d = min(k - from, NE);  // elements to drop
    const int64_t b = (int64_t)from * bits / 8;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      uint32_t w[NW];
      const uint8_t* p = row[t] + b;
#pragma unroll
      for (int i = 0; i < NW; ++i) w[i] = *reinterpret_cast<const ls_u32u*>(p + 4 * i);
      const int sh = d * bits, words = sh >> 5, rest = sh & 31;
#pragma unroll
      for (int step = 1; step < 2 * NW; step *= 2) {
#pragma unroll
        for (int i = 0; i < NW; ++i)
          w[i] = (words & step) ? (i + step < NW ? w[i + step] : 0u) : w[i];
      }
#pragma unroll
      for (int i = 0; i < NW; ++i)
        w[i] = rest ? (w[i] >> rest) | (i + 1 < NW ? w[i + 1] << (32 - rest) : 0u) : w[i];
#pragma unroll
      for (int i = 0; i < NW; ++i) r.w[t][i] = w[i];
    }
  }
  // tile t's fragment of step u
  static __device__ __forceinline__ ls_bf16x8 frag(const Regs& r, const int t, const int u) {
    constexpr int N8 = bits / 4;  // words of 8 elements
    uint32_t w[N8];
#pragma unroll
    for (int i = 0; i < N8; ++i) w[i] = r.w[t][(HALF ? 0 : u * N8) + i];
    return ls_decode8<DT>(w);
  }
  // index of the operand's element that tile t, lane row r holds
  __device__ __forceinline__ int index(const int t, int r) const { return 16 * t + r; }
  __device__ __forceinline__ bool owns(const int, int) const { return true; }
};

// Row operand of a small tile, read 64 contiguous bytes a quad of lanes: a
// memory instruction costs about a cycle per line and quad, and LsRow's lanes
// are each on a row of their own.  In block k0 (LQ_KB elements), lane (h, m, c)
// = (lane / 16, lane / 4 % 4, lane % 4) loads, for j = 0 .. 3, chunk c of K
// quarter h of row 4 m + j; a 4 x 4 transpose within each quad (two rounds of
// lane exchanges) then gives it the four chunks of row 4 m + c = lane % 16, the
// fragments' row.  Fragment step s holds elements k0 + 32 h + 8 s .. + 7.
constexpr int LQ_KB = 128;

template <int DT, int T>
struct LsQuad {
  static constexpr int bits = dtype_bits(DT);
  static constexpr int QB = 32 * bits / 8;              // bytes of a K quarter
  static constexpr int GROUPS = QB > 64 ? QB / 64 : 1;  // loads of 4 chunks a block
  static constexpr int CB = QB / GROUPS / 4;            // bytes of a chunk
  static constexpr int CW = CB / 4;                     // words
  static constexpr int STEPS = 4 / GROUPS;              // steps a group
  typedef uint32_t Chunk __attribute__((ext_vector_type(CW)));
  struct Regs {
    Chunk w[T][4];
  };
  const uint8_t* row[T][4];
  bool odd, high;

  __device__ __forceinline__ void init(const uint8_t* p, int64_t pitch, int i0, int count, int lane) {
    odd = lane & 1;
    high = lane & 2;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        row[t][j] = p + (int64_t)min(i0 + 16 * t + (lane >> 2 & 3) * 4 + j, count - 1) * pitch +
                    (lane >> 4) * QB + (lane & 3) * CB;
  }
  __device__ __forceinline__ void load(Regs& r, int k0, const int group) const {
    const int64_t b = (int64_t)k0 * bits / 8 + group * 4 * CB;
    typedef Chunk ChunkU __attribute__((aligned(1)));
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) r.w[t][j] = *reinterpret_cast<const ChunkU*>(row[t][j] + b);
  }
  template <int CTRL>
  static __device__ __forceinline__ uint32_t quad(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
  }
  // chunk j of load k <-> chunk k of load j, across the lanes of a quad
  __device__ __forceinline__ void turn(Regs& r) const {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < CW; ++i) {
        uint32_t a[4], b[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = r.w[t][j][i];
#pragma unroll
        for (int j = 0; j < 4; j += 2) {  // lanes c, c ^ 1
          const uint32_t p = quad<0xB1>(a[j + 1]), q = quad<0xB1>(a[j]);
          b[j] = odd ? p : a[j];
          b[j + 1] = odd ? a[j + 1] : q;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {     // lanes c, c ^ 2
          const uint32_t p = quad<0x4E>(b[j + 2]), q = quad<0x4E>(b[j]);
          r.w[t][j][i] = high ? p : b[j];
          r.w[t][j + 2][i] = high ? b[j + 2] : q;
        }
      }
  }
  // tile t's fragment of step s (turned)
  static __device__ __forceinline__ ls_bf16x8 frag(const Regs& r, const int t, const int s) {
    constexpr int N8 = bits / 4;  // words of 8 elements
    uint32_t w[N8];
#pragma unroll
    for (int i = 0; i < N8; ++i) {
      const int at = (s % STEPS) * N8 + i;
      w[i] = r.w[t][at / CW][at % CW];
    }
    return ls_decode8<DT>(w);
  }
};

// Col operand: T tiles, element (k, i) at row k of `pitch` bytes.
template <int DT, int T>
struct LsCol {
  static constexpr int bits = dtype_bits(DT);
  static constexpr int RB = T * bits;                 // bits of a lane's run
  static constexpr int NW = RB > 32 ? RB / 32 : 1;    // words of it
  static_assert(RB >= 8, "whole bytes a run");
  static constexpr bool HALF = true;
  typedef uint32_t Run __attribute__((ext_vector_type(NW)));
  struct Regs {
    Run w[8];
  };
  const uint8_t* base;
  int64_t pitch;
  int kl, last;

  // (count >= T)
  __device__ __forceinline__ void init(const uint8_t* p, int64_t pitch_, int i0, int count, int lane) {
    kl = (lane >> 4) * 16;
    pitch = pitch_;
    last = split_detail::col_last(T, count, i0);
    base = p + kl * pitch + (int64_t)(i0 + index(0, lane & 15)) * bits / 8;
  }
  __device__ __forceinline__ Run load_run(int64_t off) const {
    const uint8_t* p = base + off;
    if constexpr (RB >= 32) {
      typedef Run RunU __attribute__((aligned(1)));
      return *reinterpret_cast<const RunU*>(p);
    } else if constexpr (RB == 16) {
      return Run(*reinterpret_cast<const ls_u16u*>(p));
    } else {
      return Run(*p);
    }
  }
  __device__ __forceinline__ void load(Regs& r, int k0, const int u) const {
#pragma unroll
    for (int j = 0; j < 8; ++j) r.w[j] = load_run((k0 + 8 * u + j) * pitch);
  }
  __device__ __forceinline__ void load_tail(Regs& r, int k0, const int u, int K) const {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      r.w[j] = Run(0u);
      if (k0 + kl + 8 * u + j < K) r.w[j] = load_run((k0 + 8 * u + j) * pitch);
    }
  }
  static __device__ __forceinline__ ls_bf16x8 frag(const Regs& r, const int t, const int) {
    uint32_t o[4];
    if constexpr (bits == 32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = ls_pair(u2f(r.w[2 * i][t]), u2f(r.w[2 * i + 1][t]));
      return __builtin_bit_cast(ls_bf16x8, make_uint4(o[0], o[1], o[2], o[3]));
    } else {
      uint32_t w[bits / 4];  // 8 elements of tile t, K order
      if constexpr (bits == 16) {
        const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          w[i] = __builtin_amdgcn_perm(r.w[2 * i + 1][t / 2], r.w[2 * i][t / 2], sel);
      } else if constexpr (bits == 8) {
        const uint32_t sel = 0x0C0C0000u | (uint32_t)((4 + t) << 8) | (uint32_t)t;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint32_t lo = __builtin_amdgcn_perm(r.w[4 * i + 1][0], r.w[4 * i][0], sel);
          const uint32_t hi = __builtin_amdgcn_perm(r.w[4 * i + 3][0], r.w[4 * i + 2][0], sel);
          w[i] = lo | (hi << 16);
        }
      } else {
        w[0] = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) w[0] |= ((r.w[j][0] >> (4 * t)) & 0xFu) << (4 * j);
      }
      return ls_decode8<DT>(w);
    }
  }
  // A run that would pass the last index starts T before it instead, so edge
  // tiles take the same vector loads; what such a run repeats, or holds of the
  // tile before, is summed and not stored (owns).
  __device__ __forceinline__ int index(const int t, int r) const {
    return split_detail::col_index(T, last, t, r);
  }
  __device__ __forceinline__ bool owns(const int t, int r) const {
    return split_detail::col_owns(T, last, t, r);
  }
  // fp32 only: the sum of these 8 k of tile t's element, in K order
  static __device__ __forceinline__ float sum(const Regs& r, const int t) {
    static_assert(bits == 32, "fp32 operand");
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) s += u2f(r.w[j][t]);
    return s;
  }
};

template <int DT, bool COL, int T>
struct LsOperand : LsRow<DT, T> {};
template <int DT, int T>
struct LsOperand<DT, true, T> : LsCol<DT, T> {};

struct SplitGeom {
  int M, N, K;
  int64_t x_pitch, w_pitch;  // bytes between rows as stored
  int tiles_m, tiles_n;
  int n_vec;  // N % 4 == 0: 4-element stores
};

// x_sum (XCOL, fp32): x_sum[m] = sum over k of X(m, k) in fp32, made by the
// workgroups of the first tile column.
template <int XT, bool XCOL, int WT, bool WCOL, int MT, int NT, int NWV, bool QUAD>
__global__ __launch_bounds__(NWV * 64) void linear_split_kernel(
    const uint8_t* __restrict__ x, const float* __restrict__ x_scale,
    const uint8_t* __restrict__ w, const float* __restrict__ w_scale, Epilogue ep,
    void* __restrict__ y, float* __restrict__ x_sum, SplitGeom g) {
  using X = LsOperand<XT, XCOL, MT>;
  using Wt = LsOperand<WT, WCOL, NT>;
  constexpr int TN = 16 * NT;
  constexpr int LP = TN + 4;  // LDS row pitch (floats)
  __shared__ __attribute__((aligned(16))) float part[NWV * 16 * LP];

  // tile index: the blocks one XCD gets (block id mod 8) are consecutive
  // tiles, walked down M within groups of 8 tile rows so they share W
  const int T = g.tiles_m * g.tiles_n;
  const int xcd = (int)(blockIdx.x & 7), per = T >> 3, rest = T & 7;
  const int t = xcd * per + min(xcd, rest) + (int)(blockIdx.x >> 3);
  constexpr int GM = 8;
  const int group = t / (GM * g.tiles_n);
  const int first_m = group * GM;
  const int gm = min(g.tiles_m - first_m, GM);
  const int rem = t - group * GM * g.tiles_n;
  const int tn = rem / gm;
  const int m0 = (first_m + rem - tn * gm) * 16 * MT;
  const int n0 = tn * TN;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  X xo;
  Wt wo;
  xo.init(x, g.x_pitch, m0, g.M, lane);
  wo.init(w, g.w_pitch, n0, g.N, lane);

  ls_f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = ls_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float xs[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) xs[i] = 0.0f;
  const bool sums = XCOL && x_sum && n0 == 0;

  // blocks of this kernel's size; what is left of K goes 64 at a time
  constexpr int KB = QUAD ? LQ_KB : LS_KB;
  const int whole = g.K / KB, blocks = whole + (g.K % KB != 0);
  const int b0 = (int)((int64_t)blocks * wave / NWV), b1 = (int)((int64_t)blocks * (wave + 1) / NWV);
  const int e = min(b1, whole);
  // One MFMA step: half u of a block.
  auto multiply = [&](const typename X::Regs& rx, const typename Wt::Regs& rw, const int u) {
    ls_bf16x8 a[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) a[j] = Wt::frag(rw, j, u);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const ls_bf16x8 b = X::frag(rx, i, u);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j], b, acc[i][j], 0, 0, 0);
    }
    if constexpr (XCOL && XT == F32) {
      if (sums) {
#pragma unroll
        for (int i = 0; i < MT; ++i) xs[i] += X::sum(rx, i);
      }
    }
  };
  // the last K elements from k0, fewer than a 64-K block
  auto tail = [&](typename X::Regs& rx, typename Wt::Regs& rw, int k0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (u == 0 || X::HALF) xo.load_tail(rx, k0, u, g.K);
      if (u == 0 || Wt::HALF) wo.load_tail(rw, k0, u, g.K);
      multiply(rx, rw, u);
    }
  };
  const bool ragged = b1 > whole && b0 < b1;  // this wave has the ragged last block
  // Two register sets an operand, the next one's loads in flight while a step
  // multiplies.
  if constexpr (QUAD) {
    using Q = LsQuad<XT, MT>;
    using R = LsQuad<WT, NT>;
    Q xq;
    R wq;
    xq.init(x, g.x_pitch, m0, g.M, lane);
    wq.init(w, g.w_pitch, n0, g.N, lane);
    typename Q::Regs qx[2];
    typename R::Regs qw[2];
    static_assert(R::GROUPS == 1, "weights of 16 bits and fewer");
    // Block b, whose first x group (and whole block, in set P) is loaded already.
    auto block = [&](int b, const int P) {
      const bool next = b + 1 < e;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const int px = Q::GROUPS == 2 ? s >> 1 : P;
        if constexpr (Q::GROUPS == 2) {
          if (s == 0) xq.load(qx[1], b * LQ_KB, 1);
          if (s == 2 && next) xq.load(qx[0], (b + 1) * LQ_KB, 0);
        } else {
          if (s == 0 && next) xq.load(qx[P ^ 1], (b + 1) * LQ_KB, 0);
        }
        if (s == 0) {
          if (next) wq.load(qw[P ^ 1], (b + 1) * LQ_KB, 0);
          wq.turn(qw[P]);
        }
        if (s % Q::STEPS == 0) xq.turn(qx[px]);
        ls_bf16x8 a[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) a[j] = R::frag(qw[P], j, s);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const ls_bf16x8 v = Q::frag(qx[px], i, s);
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j], v, acc[i][j], 0, 0, 0);
        }
      }
    };
    if (b0 < e) {
      xq.load(qx[0], b0 * LQ_KB, 0);
      wq.load(qw[0], b0 * LQ_KB, 0);
    }
    for (int b = b0; b < e; b += 2) {
      block(b, 0);
      if (b + 1 < e) block(b + 1, 1);
    }
    if (ragged) {
      typename X::Regs rx;
      typename Wt::Regs rw;
      int k0 = whole * LQ_KB;
      if (k0 + LS_KB <= g.K) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          if (u == 0 || X::HALF) xo.load(rx, k0, u);
          if (u == 0 || Wt::HALF) wo.load(rw, k0, u);
          multiply(rx, rw, u);
        }
        k0 += LS_KB;
      }
      if (k0 < g.K) tail(rx, rw, k0);
    }
  } else {
    typename X::Regs rx[2];
    typename Wt::Regs rw[2];
    // Block b, whose first half (and whole codes, in set P) is loaded already.
    auto block = [&](int b, const int P) {
      if constexpr (X::HALF) xo.load(rx[1], b * LS_KB, 1);
      if constexpr (Wt::HALF) wo.load(rw[1], b * LS_KB, 1);
      multiply(rx[X::HALF ? 0 : P], rw[Wt::HALF ? 0 : P], 0);
      if (b + 1 < e) {
        xo.load(rx[X::HALF ? 0 : P ^ 1], (b + 1) * LS_KB, 0);
        wo.load(rw[Wt::HALF ? 0 : P ^ 1], (b + 1) * LS_KB, 0);
      }
      multiply(rx[X::HALF ? 1 : P], rw[Wt::HALF ? 1 : P], 1);
    };
    if (b0 < e) {
      xo.load(rx[0], b0 * LS_KB, 0);
      wo.load(rw[0], b0 * LS_KB, 0);
    }
    for (int b = b0; b < e; b += 2) {
      block(b, 0);
      if (b + 1 < e) block(b + 1, 1);
    }
    if (ragged) tail(rx[0], rw[0], whole * LS_KB);
  }

  // add the waves' tiles in wave order, 16 rows of X (one MT tile) at a time
  const float s = product_scale(w_scale, x_scale);
  const float inv_o = epi_inv_scale(ep);
  uint32_t am = 0;
  const int q4 = (lane >> 4) * 4;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    if (i) __syncthreads();
    float* mine = part + (wave * 16 + (lane & 15)) * LP;
    if constexpr (WCOL) {
      // a lane's NT tiles are consecutive n
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          if (wo.owns(j, q4 + q)) mine[wo.index(j, q4 + q)] = acc[i][j][q];
    } else {
#pragma unroll
      for (int j = 0; j < NT; ++j) *reinterpret_cast<ls_f32x4*>(mine + 16 * j + q4) = acc[i][j];
    }
    __syncthreads();
    for (int o = tid; o < 16 * TN / 4; o += NWV * 64) {
      const int r = o / (TN / 4), c = (o - r * (TN / 4)) * 4;
      const int m = m0 + xo.index(i, r), n = n0 + c;
      if (m >= g.M || n >= g.N || !xo.owns(i, r)) continue;
      ls_f32x4 v = *reinterpret_cast<const ls_f32x4*>(part + r * LP + c);
#pragma unroll
      for (int k = 1; k < NWV; ++k)
        v = v + *reinterpret_cast<const ls_f32x4*>(part + (k * 16 + r) * LP + c);
      float f[4];
      const int live = min(4, g.N - n);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (k >= live) break;
        f[k] = epi_value(ep, epi_chan(ep, n + k), v[k], s);
        if (ep.amax) am = epi_track(am, f[k]);
      }
      const int64_t at = (int64_t)m * g.N + n;
      if (g.n_vec) {
        epi_store4(ep.out_dtype, y, at, f, inv_o);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k < live) epi_store(ep.out_dtype, y, at + k, f[k], inv_o);
      }
    }
  }
  epi_amax_commit(ep, am);

  if constexpr (XCOL && XT == F32) {
    if (sums) {
      // lanes r, r + 16, r + 32, r + 48 hold the same columns' K quarters
      __syncthreads();
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        float v = xs[i];
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (lane < 16 && xo.owns(i, lane)) part[wave * 16 * MT + xo.index(i, lane)] = v;
      }
      __syncthreads();
      for (int o = tid; o < 16 * MT; o += NWV * 64) {
        if (m0 + o >= g.M) continue;
        float v = part[o];
#pragma unroll
        for (int k = 1; k < NWV; ++k) v += part[k * 16 * MT + o];
        x_sum[m0 + o] = v;
      }
    }
  }
}

template <int XT, bool XCOL, int WT, bool WCOL, int MT, int NT, int NWV, bool QUAD = false>
int split_launch_tile(const uint8_t* x, const float* x_scale, const uint8_t* w,
                      const float* w_scale, const Epilogue& ep, void* y, float* x_sum,
                      SplitGeom g, hipStream_t stream) {
  const int64_t tm = ((int64_t)g.M + 16 * MT - 1) / (16 * MT);
  const int64_t tn = ((int64_t)g.N + 16 * NT - 1) / (16 * NT);
  if (tm * tn > 0x7FFFFFFF) return NOVAQ_EINVAL;
  g.tiles_m = (int)tm;
  g.tiles_n = (int)tn;
  hipLaunchKernelGGL((linear_split_kernel<XT, XCOL, WT, WCOL, MT, NT, NWV, QUAD>),
                     dim3((unsigned)(tm * tn)), dim3(NWV * 64), 0, stream, x, x_scale, w, w_scale,
                     ep, y, x_sum, g);
  return check_launch();
}

// Pitches in bytes of the operands as stored: row operands are (M or N) x K,
// col operands K x (M or N).
template <int XT, bool XCOL, int WT, bool WCOL>
int split_launch(const uint8_t* x, const float* x_scale, int64_t M, int64_t K, const uint8_t* w,
                 const float* w_scale, const Epilogue& ep, int64_t N, void* y, float* x_sum,
                 hipStream_t stream) {
  if (M > 0x7FFFFFFF || N > 0x7FFFFFFF || K > 0x7FFFFFFF) return NOVAQ_EINVAL;
  SplitGeom g{};
  g.M = (int)M;
  g.N = (int)N;
  g.K = (int)K;
  g.x_pitch = ((XCOL ? M : K) * dtype_bits(XT) + 7) / 8;
  g.w_pitch = ((WCOL ? N : K) * dtype_bits(WT) + 7) / 8;
  g.n_vec = N % 4 == 0;
  const int64_t tiles64 = ((M + 63) / 64) * ((N + 63) / 64);
  if constexpr (!XCOL && !WCOL) {
    // Lines read whole by quads of lanes (LsQuad) halve a long product's time
    // (64 x 4096 x 4096, bf16 x, FP4 W: 9.6 us against 14.7).  Its larger blocks
    // and registers need waves with work for them: from 4 rows (2 rows 7.5 us
    // against 7.3), 2048 K over 16 waves (1024: 5.0, 4.5), and with one
    // workgroup a CU 512 K over 8 (128 x 256 x 256: 5.5, 4.8; 64 x 2048 x 513:
    // 6.0, 8.3), with more 1024 K without a rest (1000 x 500 x 784: 15.2, 11.4;
    // 500 x 1024 x 1024: 8.9, 9.4) or 2048.  Over 3990 products of 1 to 1000 rows, K
    // 256 to 4096 and 256 to 4096 columns (E4M3 and FP4 W, fp32 and bf16 x), each
    // run both ways, these lines are 0.8% from the better one on average and more
    // than a fifth on 27, all of them a K of 2100 or 3000 with several workgroups a
    // CU, or 1536 with at most 16 rows; without quads 5.9%, with them wherever they
    // can run 6.4%.
    if constexpr (dtype_bits(WT) <= 16) {
      const int64_t tiles32 = ((M + 31) / 32) * ((N + 31) / 32);
      if (M >= 4 && M <= 16 && K >= 2048)
        return split_launch_tile<XT, XCOL, WT, WCOL, 1, 1, 16, true>(x, x_scale, w, w_scale, ep, y, x_sum, g, stream);
      if (M > 16 && tiles64 < device_cu_count() &&
          (K >= 2048 || (tiles32 <= device_cu_count() ? K >= 512 : K >= 1024 && K % LQ_KB == 0)))
        return split_launch_tile<XT, XCOL, WT, WCOL, 2, 2, 8, true>(x, x_scale, w, w_scale, ep, y, x_sum, g, stream);
    }
    if (M <= 16)
      return split_launch_tile<XT, XCOL, WT, WCOL, 1, 1, 16>(x, x_scale, w, w_scale, ep, y, x_sum, g, stream);
  }
  // (two fp32 col operands: 64 x 32, the registers of 64 x 64 would spill)
  constexpr int BIG_NT = XCOL && WCOL ? 2 : 4;
  if (tiles64 >= device_cu_count())
    return split_launch_tile<XT, XCOL, WT, WCOL, 4, BIG_NT, 4>(x, x_scale, w, w_scale, ep, y, x_sum, g, stream);
  return split_launch_tile<XT, XCOL, WT, WCOL, 2, 2, 8>(x, x_scale, w, w_scale, ep, y, x_sum, g, stream);
}

}  // namespace
}  // namespace novaq
