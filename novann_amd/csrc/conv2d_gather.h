// Conv2d on bf16 MFMA with the input window gathered straight into fragment
// registers (gfx950): zeros padding, any channel count and stride, for shapes
// whose input rows do not fit or do not pay to be staged in LDS.
//
// GEMM view: M = output channels, N = output pixels of the whole batch (so
// maps of any size fill the tiles), K = (c, kh, kw) in the weights' own order,
// so a weight row is a K-contiguous operand of linear_split.h and is read from
// memory as stored.  The pixel operand is gathered: element (k, p) is
// x[base(p) + off(k)], where off is an LDS table the workgroup makes once and
// base and a bit mask of the taps inside the image are worked out once per
// lane and pixel tile.  A tap outside the image turns the load's offset into
// one past the buffer descriptor, which returns 0, the padding: four
// instructions an element and no branch.
//
// A wave's tile is 16 MT channels x 16 NT pixels.  Its 4 waves take either 4
// neighbouring pixel tiles (many tiles) or a quarter of K each of one tile (few tiles: more waves in flight).  What bounds it: the
// gather's vector instructions and 4-byte loads, shared by the tile's
// channels, so MT is as large as C_out fills (128 channels x 32 pixels a wave
// for more than 64).  Measured (E4M3 weights, fp32 x, warm MALL): 64 -> 128
// channels, 3 x 3 / 2, 256 maps of 28 x 28: 45.7 us, 3714 on the one-lane-an-
// output kernel it took over from; 128 -> 128, 3 x 3, 64 maps of 14 x 14: 22.7
// us, 81.2 on conv2d_kernel; one 64 -> 128 map of 28 x 28: 9.3 us, 20.5 on the
// band kernel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "linear_split.h"
#include "novaq_convert.h"
#include "novaq_epilogue.h"
#include "novaq_internal.h"
#include "novaq_xload.h"

namespace novaq {
namespace {

constexpr int CG_TAP_SHIFT = 26;                       // table entry: tap, offset
constexpr uint32_t CG_OFF_MASK = (1u << CG_TAP_SHIFT) - 1;
constexpr int CG_MAX_TAPS = 31;                        // tap 31: always outside (K padding)
constexpr int CG_MAX_K = 16 * 1024;                    // table entries

struct GatherGeom {
  int M;                // rows: output channels of this product
  int K;                // gathered channels * taps
  int taps, KH, KW;
  int GH, GW;           // gathered image
  int PH, PW;           // output pixels of an image
  int sh, sw, ph, pw;
  int gathered;         // elements of one gathered image (channels * GH * GW)
  int images;           // N
  int64_t pixels;       // N * PH * PW
  int64_t w_pitch;      // bytes of a weight row
  int tiles_m, tiles_n; // workgroup tiles
  int ksplit;           // the waves split K (else neighbouring pixel tiles)
  int quads;            // PH * PW % 4 == 0: 4 consecutive pixels share an image
  FastDiv fd_taps, fd_kw, fd_pp, fd_pw;
};

template <int XT, int NT>
struct CgPixels {
  static constexpr int XB = XL<XT>::bytes;
  struct Regs {
    uint32_t w[NT][8];
  };
  __amdgpu_buffer_rsrc_t rs;
  const uint32_t* tab;   // this lane group's entries of block 0
  uint32_t base[NT];
  uint32_t outside[NT];  // bit t: tap t is outside the image

  // pixels p0 .. p0 + 16 NT - 1 (clamped to the last one)
  __device__ __forceinline__ void init(const uint8_t* x, const uint32_t* table, int p0, int lane,
                                       const GatherGeom& g) {
    tab = table + (lane >> 4) * 16;
    const int last = (int)g.pixels - 1;
    const int n0 = __builtin_amdgcn_readfirstlane((int)fdiv((uint32_t)min(p0, last), g.fd_pp));
    const int64_t left = (int64_t)(g.images - n0) * g.gathered * XB;
    rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(x + (int64_t)n0 * g.gathered * XB),
                                           (short)0, (int)(left < 0x7FFFFFFF ? left : 0x7FFFFFFF),
                                           0x00020000);
    const int pp = g.PH * g.PW;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int p = min(p0 + 16 * t + (lane & 15), last);
      const int n = (int)fdiv((uint32_t)p, g.fd_pp), q = p - n * pp;
      const int oy = (int)fdiv((uint32_t)q, g.fd_pw), ox = q - oy * g.PW;
      const int y0 = oy * g.sh - g.ph, x0 = ox * g.sw - g.pw;
      const int lo = min(max(0, -x0), g.KW), hi = max(min(g.KW, g.GW - x0), 0);
      const uint32_t cols = hi > lo ? ((1u << hi) - 1u) & ~((1u << lo) - 1u) : 0u;
      uint32_t in = 0;
      for (int a = 0; a < g.KH; ++a)
        if ((unsigned)(y0 + a) < (unsigned)g.GH) in |= cols << (a * g.KW);
      outside[t] = ~in;
      base[t] = (uint32_t)((n - n0) * g.gathered + y0 * g.GW + x0);
    }
  }
  __device__ __forceinline__ void load(Regs& r, int k0, const int u) const {
    const uint4 a = *reinterpret_cast<const uint4*>(tab + k0 + 8 * u);
    const uint4 b = *reinterpret_cast<const uint4*>(tab + k0 + 8 * u + 4);
    const uint32_t e[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t tap = e[j] >> CG_TAP_SHIFT, off = e[j] & CG_OFF_MASK;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint32_t miss = (uint32_t)__builtin_amdgcn_sbfe((int)outside[t], tap, 1u);
        const uint32_t at = ((base[t] + off) * XB) | (miss & 0x80000000u);
        if constexpr (XB == 4) r.w[t][j] = __builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0);
        else if constexpr (XB == 2) r.w[t][j] = __builtin_amdgcn_raw_buffer_load_b16(rs, at, 0, 0);
        else r.w[t][j] = __builtin_amdgcn_raw_buffer_load_b8(rs, at, 0, 0);
      }
    }
  }
  static __device__ __forceinline__ ls_bf16x8 frag(const Regs& r, const int t) {
    if constexpr (XB == 4) {
      return ls_decode8<XT>(r.w[t]);
    } else if constexpr (XB == 2) {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = r.w[t][2 * i] | (r.w[t][2 * i + 1] << 16);
      return ls_decode8<XT>(w);
    } else {
      uint32_t w[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        w[i] = r.w[t][4 * i] | (r.w[t][4 * i + 1] << 8) | (r.w[t][4 * i + 2] << 16) |
               (r.w[t][4 * i + 3] << 24);
      return ls_decode8<XT>(w);
    }
  }
};

template <int WT, int XT, int MT, int NT>
__global__ __launch_bounds__(256, 2) void conv2d_gather_kernel(
    const uint8_t* __restrict__ x, const float* __restrict__ x_scale,
    const uint8_t* __restrict__ w, const float* __restrict__ w_scale, Epilogue ep,
    void* __restrict__ y, GatherGeom g) {
  using Px = CgPixels<XT, NT>;
  using Wt = LsRow<WT, MT>;
  constexpr int TN = 16 * NT;
  extern __shared__ __attribute__((aligned(16))) uint32_t cg_lds[];
  uint32_t* tab = cg_lds;     // K rounded up to whole blocks
  const int blocks = (g.K + LS_KB - 1) / LS_KB, whole = g.K / LS_KB;

  // tile index: the blocks one XCD gets (block id mod 8) are consecutive
  // tiles, the channel blocks of one pixel tile next to each other
  const int T = g.tiles_m * g.tiles_n;
  const int xcd = (int)(blockIdx.x & 7), per = T >> 3, rest = T & 7;
  const int t = xcd * per + min(xcd, rest) + (int)(blockIdx.x >> 3);
  const int tn = t / g.tiles_m;
  const int m0 = (t - tn * g.tiles_m) * 16 * MT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p0 = (g.ksplit ? tn : 4 * tn + wave) * TN;

  for (int k = tid; k < blocks * LS_KB; k += 256) {
    uint32_t e = 31u << CG_TAP_SHIFT;
    if (k < g.K) {
      const int c = (int)fdiv((uint32_t)k, g.fd_taps), tap = k - c * g.taps;
      const int a = (int)fdiv((uint32_t)tap, g.fd_kw), b = tap - a * g.KW;
      const int off = c * (g.GH * g.GW) + a * g.GW + b;
      e = ((uint32_t)tap << CG_TAP_SHIFT) | (uint32_t)off;
    }
    tab[k] = e;
  }
  Px px;
  Wt wo;
  px.init(x, tab, p0, lane, g);
  wo.init(w, g.w_pitch, m0, g.M, lane);
  __syncthreads();

  ls_f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = ls_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  const int b0 = g.ksplit ? blocks * wave / 4 : 0, b1 = g.ksplit ? blocks * (wave + 1) / 4 : blocks;
  auto multiply = [&](const typename Px::Regs& rx, const typename Wt::Regs& rw, const int u) {
    ls_bf16x8 a[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) a[j] = Px::frag(rx, j);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const ls_bf16x8 b = Wt::frag(rw, i, u);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j], b, acc[i][j], 0, 0, 0);
    }
  };
  // two register sets an operand, as in linear_split_kernel; the gather's
  // table covers the ragged last block, the weights' rows do not
  typename Px::Regs rx[2];
  typename Wt::Regs rw[2];
  auto load_w = [&](typename Wt::Regs& r, int b, const int u) {
    if (b < whole) wo.load(r, b * LS_KB, u);
    else wo.load_end(r, b * LS_KB, u, g.K);
  };
  auto block = [&](int b, const int P) {
    px.load(rx[1], b * LS_KB, 1);
    if constexpr (Wt::HALF) load_w(rw[1], b, 1);
    multiply(rx[0], rw[Wt::HALF ? 0 : P], 0);
    if (b + 1 < b1) {
      px.load(rx[0], (b + 1) * LS_KB, 0);
      load_w(rw[Wt::HALF ? 0 : P ^ 1], b + 1, 0);
    }
    multiply(rx[1], rw[Wt::HALF ? 1 : P], 1);
  };
  if (b0 < b1) {
    px.load(rx[0], b0 * LS_KB, 0);
    load_w(rw[0], b0, 0);
  }
  for (int b = b0; b < b1; b += 2) {
    block(b, 0);
    if (b + 1 < b1) block(b + 1, 1);
  }

  // The workgroup's outputs meet in LDS: its 4 neighbouring pixel tiles side by
  // side, or the one tile's K quarters added pairwise, (0 + 2) + (1 + 3).
  // One loop then stores runs of 4 pixels (a single copy of the epilogue, and
  // consecutive lanes on consecutive runs of a channel).
  const float s = product_scale(w_scale, x_scale);
  const float inv_o = epi_inv_scale(ep), z = epi_relu_factor(ep);
  float* out = reinterpret_cast<float*>(tab);
  const int q4 = (lane >> 4) * 4, rl = lane & 15;
  const int cols = g.ksplit ? TN : 4 * TN, pitch = cols + 4;
  auto put = [&](float* d) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        *reinterpret_cast<ls_f32x4*>(d + (16 * i + rl) * pitch + 16 * j + q4) = acc[i][j];
  };
  auto add = [&](const float* d) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = acc[i][j] +
                    *reinterpret_cast<const ls_f32x4*>(d + (16 * i + rl) * pitch + 16 * j + q4);
  };
  __syncthreads();  // every wave is done with the table
  if (g.ksplit) {
    float* half = out + (wave & 1) * 16 * MT * pitch;
    if (wave >= 2) put(half);
    __syncthreads();
    if (wave < 2) add(half);
    if (wave == 1) put(half);
    __syncthreads();
    if (wave == 0) {
      add(out + 16 * MT * pitch);
      put(out);
    }
  } else {
    put(out + wave * TN);
  }
  __syncthreads();
  const int pp = g.PH * g.PW;
  const int first = tn * cols;  // the workgroup's first pixel
  const int runs = cols / 4;
  uint32_t am = 0;
  for (int o = tid; o < 16 * MT * runs; o += 256) {
    const int r = o / runs, c = (o - r * runs) * 4;
    const int co = m0 + r, p = first + c, live = (int)g.pixels - p;
    if (co >= g.M || live <= 0) continue;
    const ls_f32x4 v = *reinterpret_cast<const ls_f32x4*>(out + r * pitch + c);
    const EpiChan k = epi_chan(ep, co);
    float f[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f[q] = epi_value_nb(k, v[q], s, z);
      if (q < live) am = epi_track(am, f[q]);
    }
    if (g.quads) {
      const int n = (int)fdiv((uint32_t)p, g.fd_pp);
      epi_store4(ep.out_dtype, y, ((int64_t)n * g.M + co) * pp + (p - n * pp), f, inv_o);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q >= live) break;
        const int n = (int)fdiv((uint32_t)(p + q), g.fd_pp);
        epi_store(ep.out_dtype, y, ((int64_t)n * g.M + co) * pp + (p + q - n * pp), f[q], inv_o);
      }
    }
  }
  epi_amax_commit(ep, am);
}

template <int WT, int XT, int MT, int NT>
int gather_launch_tile(const uint8_t* x, const float* x_scale, const uint8_t* w,
                       const float* w_scale, const Epilogue& ep, void* y, GatherGeom g,
                       hipStream_t stream) {
  constexpr int TN = 16 * NT;
  const int64_t tm = ((int64_t)g.M + 16 * MT - 1) / (16 * MT);
  const int64_t wave_tiles = (g.pixels + TN - 1) / TN;
  // neighbouring pixel tiles a wave once that still gives each CU two
  // workgroups
  g.ksplit = tm * wave_tiles < (int64_t)8 * device_cu_count();
  const int64_t tn = g.ksplit ? wave_tiles : (wave_tiles + 3) / 4;
  if (tm * tn > 0x7FFFFFFF) return NOVAQ_ENOTSUP;
  g.tiles_m = (int)tm;
  g.tiles_n = (int)tn;
  const size_t table = (size_t)((g.K + LS_KB - 1) / LS_KB) * LS_KB * 4;
  const size_t out = (size_t)16 * MT * (g.ksplit ? 2 * (TN + 4) : 4 * TN + 4) * 4;
  const size_t lds = table > out ? table : out;
  constexpr size_t MOST = 16 * MT * (4 * TN + 4) * 4 > CG_MAX_K * 4 ? 16 * MT * (4 * TN + 4) * 4
                                                                    : CG_MAX_K * 4;
  static DeviceFlags raised;  // per instantiation
  auto kern = conv2d_gather_kernel<WT, XT, MT, NT>;
  const int rc = allow_lds(raised, reinterpret_cast<const void*>(kern), lds, MOST);
  if (rc != NOVAQ_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(tm * tn)), dim3(256), lds, stream, x, x_scale, w,
                     w_scale, ep, y, g);
  return check_launch();
}

// Whether the kernel takes the product at all: zeros padding is the caller's
// to check.  `gathered` elements per gathered image, taps = KH * KW.
template <int WT, int XT>
bool gather_takes(int64_t M, int64_t channels, int64_t GH, int64_t GW, int64_t taps,
                  int64_t images, int64_t pp) {
  const int64_t K = channels * taps, gathered = channels * GH * GW;
  if (taps > CG_MAX_TAPS || K < 16 || K > CG_MAX_K || M > 0x7FFFFFFF) return false;
  if (dtype_bits(WT) == 4 && K % 2) return false;  // rows of whole bytes
  if (gathered + (int64_t)32 * GW >= (int64_t)1 << CG_TAP_SHIFT) return false;
  if (images * pp >= 0x7FFFFFFF - 1024) return false;
  // a wave's 64 pixels reach this many images past its first one
  const int64_t span = 64 / pp + 2;
  return span * gathered * XL<XT>::bytes < 0x7FFFFFFF;
}

template <int WT, int XT>
int gather_launch(const uint8_t* x, const float* x_scale, const uint8_t* w, const float* w_scale,
                  const Epilogue& ep, void* y, GatherGeom g, hipStream_t stream) {
  g.taps = g.KH * g.KW;
  g.w_pitch = (int64_t)g.K * dtype_bits(WT) / 8;
  g.pixels = (int64_t)g.images * g.PH * g.PW;
  g.quads = g.PH * g.PW % 4 == 0;
  g.fd_taps = fast_div((uint32_t)g.taps);
  g.fd_kw = fast_div((uint32_t)g.KW);
  g.fd_pp = fast_div((uint32_t)(g.PH * g.PW));
  g.fd_pw = fast_div((uint32_t)g.PW);
  // (fp32 weights: the registers of 8 channel tiles would spill)
  constexpr int MT_BIG = WT == F32 ? 4 : 8, NT_BIG = WT == F32 ? 4 : 2;
  if (g.M > 64) return gather_launch_tile<WT, XT, MT_BIG, NT_BIG>(x, x_scale, w, w_scale, ep, y, g, stream);
  if (g.M > 32) return gather_launch_tile<WT, XT, 4, 4>(x, x_scale, w, w_scale, ep, y, g, stream);
  return gather_launch_tile<WT, XT, 2, 4>(x, x_scale, w, w_scale, ep, y, g, stream);
}

}  // namespace
}  // namespace novaq
