// Conv2d on bf16 MFMA with the input staged channel-last in chunks of 32
// channels (gfx950): zeros padding, 3 x 3 and 1 x 1 windows, FP8 / FP4
// weights, C a multiple of 32, any stride.
//
// A workgroup of 4 waves owns a band of whole output rows of one image -- or
// several whole images where maps are small -- and 16 NCO WCO output channels;
// a wave owns 64 of its pixels and 16 NCO channels (WCO waves side by side in
// channels, the rest in pixels): 4 x NCO accumulators of
// v_mfma_f32_16x16x32_bf16 with pixels as rows, so 4 LDS reads of x and NCO of
// weights feed 4 NCO products.  K runs chunk by chunk, one tap's 32 channels
// a step:
//   - x: the band's input rows are one contiguous run of each channel plane, so
//     an item is 4 consecutive elements of 8 planes (loads at any element
//     boundary; a run's last item starts 4 before its end instead of passing
//     it), rounded to bf16 and written as 4 x 16 bytes to [row][col][32]; the
//     border of the region is zeroed once;
//   - weights: a lane takes the 8 channels x taps of one output channel, whose
//     codes are consecutive, and regroups them with constant byte selects to
//     [tap][co][32 channels], packed codes decoded per fragment.
// The next chunk's loads go to registers before the current chunk's products
// and are written to LDS after them.  Bound by a chunk's load latency and the
// LDS traffic beside the MFMAs, the workgroups of a CU overlapping each other
// (64 -> 128, 3 x 3 / 2, and 64 -> 32 on maps of 28 x 28, 128 -> 128 on 14 x 14:
// waves wait 37-46% of their time, the LDS is busy 34-40% and half of that are
// bank conflicts, the MFMAs 13-21%).
// Measured (E4M3, fp32 x, warm MALL; the kernels it took over from in
// brackets): 64 -> 128 channels, 3 x 3 / 2, 256 maps of 28 x 28 27.1 us
// (gathered 45.9), 256 -> 256 on 256 maps of 7 x 7 36.3 (gathered 69.9), 64 ->
// 64 on 32 maps of 56 x 56 23.8 (gathered 40.6), 64 -> 64 on 256 maps of 28 x
// 28 34.5 (bands 58.5; FP4 31.9, bands 34.7).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "linear_split.h"
#include "novaq_convert.h"
#include "novaq_epilogue.h"
#include "novaq_internal.h"
#include "novaq_xload.h"

namespace novaq {
namespace {

constexpr int CK_C = 32;        // channels a chunk
// bf16 per staged pixel: fragment reads of 16 neighbours in a row meet no bank
// twice (strided pixels, row ends and the staging writes do)
constexpr int CK_PS = CK_C + 8;

struct ChunkGeom {
  int N, C, H, W, M, KH, KW, sh, sw, ph, pw, OH, OW;
  int R, bands;      // output rows of a band, bands of an image
  int G;             // images of a workgroup (bands == 1 when above 1)
  int P;             // pixels of a band: R * OW
  int rows_in, cols; // staged region of an image
  int nit;           // 4-element items of the longest run
  int tiles_m, groups;  // channel blocks; image groups
  int vec4;          // P and OH * OW multiples of 4: runs of 4 pixels are stored whole
  int x_bytes;       // staged x (the weights follow)
  FastDiv fd_w, fd_ow, fd_p, fd_nit;
};

// Words of a lane's 8 channels x T taps of codes.
template <int WT, int T>
constexpr int ck_words() { return 8 * T * dtype_bits(WT) / 32; }

// Tap t's 8 codes from the run (code of channel j at j * T + t), t constant.
template <int WT, int T>
__device__ __forceinline__ void ck_tap(const uint32_t* w, const int t, uint32_t* o) {
  if constexpr (T == 1) {
#pragma unroll
    for (int i = 0; i < ck_words<WT, T>(); ++i) o[i] = w[i];
  } else if constexpr (dtype_bits(WT) == 8) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t p[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int a = (4 * h + 2 * q) * T + t, b = a + T;
        p[q] = __builtin_amdgcn_perm(w[b >> 2], w[a >> 2],
                                     0x0C0C0000u | (uint32_t)((4 + (b & 3)) << 8) | (uint32_t)(a & 3));
      }
      o[h] = p[0] | (p[1] << 16);
    }
  } else {
    uint32_t v = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int e = j * T + t;
      v |= ((w[e >> 3] >> (4 * (e & 7))) & 0xFu) << (4 * j);
    }
    o[0] = v;
  }
}

template <int WT, int XT, int T, int NCO, int WCO, int IPT>
__global__ __launch_bounds__(256, 2) void conv2d_chunk_kernel(
    const uint8_t* __restrict__ x, const float* __restrict__ x_scale,
    const uint8_t* __restrict__ w, const float* __restrict__ w_scale, Epilogue ep,
    void* __restrict__ y, ChunkGeom g) {
  constexpr int NPX = 4;                    // pixel tiles of a wave
  constexpr int COB = 16 * NCO * WCO;       // channels of the workgroup
  constexpr int WPX = 4 / WCO;              // waves along pixels
  constexpr int NPIX = 16 * NPX * WPX;      // pixel slots of the workgroup
  constexpr int XB = XL<XT>::bytes;
  constexpr int GB = dtype_bits(WT);        // bytes of 8 codes
  constexpr int WW = ck_words<WT, T>();
  constexpr int RUNS = COB * 4 / 256;       // weight runs of a lane
  static_assert(RUNS >= 1 || COB * 4 == 128, "weight runs");
  constexpr int NR = RUNS < 1 ? 1 : RUNS;
  extern __shared__ __attribute__((aligned(16))) uint8_t ck_lds[];
  uint16_t* xl = reinterpret_cast<uint16_t*>(ck_lds);
  uint8_t* wl = ck_lds + g.x_bytes;

  // blocks of one XCD (block id mod 8) take neighbouring tiles, a band's
  // channel blocks next to each other
  const int total = g.tiles_m * g.groups * g.bands;
  const int xcd = (int)(blockIdx.x & 7), per = total >> 3, rem = total & 7;
  const int t0 = xcd * per + min(xcd, rem) + (int)(blockIdx.x >> 3);
  const int pt = t0 / g.tiles_m;
  const int co0 = (t0 - pt * g.tiles_m) * COB;
  const int grp = pt / g.bands, band = pt - grp * g.bands;
  const int n0 = grp * g.G, images = min(g.G, g.N - n0);
  const int oh0 = band * g.R, rows = min(g.R, g.OH - oh0);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int wpx = wave % WPX, wco = wave / WPX;

  // the input rows of the band: a run of L elements of each plane
  const int ih0 = oh0 * g.sh - g.ph;
  const int lo = max(ih0, 0), hi = min(ih0 + g.rows_in, g.H);
  const int L = max(0, (hi - lo) * g.W);
  const int64_t HW = (int64_t)g.H * g.W;
  const int region = g.rows_in * g.cols;    // staged pixels of an image
  const int items = images * 4 * g.nit;

  struct Item {
    uint32_t v[8][XB == 4 ? 4 : (XB == 2 ? 2 : 1)];
  };
  Item xr[IPT];
  uint32_t wr[NR][WW];
  auto load_x = [&](int c0) {
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
      // (no load behind a branch: lanes without an item repeat the last one)
      const int it = min(tid + 256 * k, items - 1);
      const int so = (int)fdiv((uint32_t)it, g.fd_nit), i = it - so * g.nit;
      const int e = max(0, min(4 * i, L - 4));
      const int64_t at = ((int64_t)(n0 + (so >> 2)) * g.C + c0 + 8 * (so & 3)) * HW +
                         (int64_t)min(lo, g.H - 1) * g.W + e;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint8_t* p = x + (at + j * HW) * XB;
        if constexpr (XB == 4) {
          const ls_u32x4u v = *reinterpret_cast<const ls_u32x4u*>(p);
#pragma unroll
          for (int q = 0; q < 4; ++q) xr[k].v[j][q] = v[q];
        } else if constexpr (XB == 2) {
          const ls_u32x2u v = *reinterpret_cast<const ls_u32x2u*>(p);
          xr[k].v[j][0] = v[0];
          xr[k].v[j][1] = v[1];
        } else {
          xr[k].v[j][0] = *reinterpret_cast<const ls_u32u*>(p);
        }
      }
    }
  };
  auto store_x = [&]() {
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
      const int it = tid + 256 * k;
      const int so = (int)fdiv((uint32_t)it, g.fd_nit), i = it - so * g.nit;
      if (it >= items || 4 * i >= L) continue;
      const int e = min(4 * i, L - 4);
      int r = (int)fdiv((uint32_t)e, g.fd_w), c = e - r * g.W;
      // channel pairs of the four elements, as bf16
      uint32_t o[4][4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t* a = xr[k].v[2 * j];
        const uint32_t* b = xr[k].v[2 * j + 1];
        if constexpr (XT == F32) {
#pragma unroll
          for (int q = 0; q < 4; ++q) o[q][j] = ls_pair(u2f(a[q]), u2f(b[q]));
        } else {
          // (element 2 i, 2 i + 1) pairs of each plane, then the two planes'
          // halves regrouped by element
          xl_u32x4 ra = {a[0], XB == 2 ? a[XB == 2 ? 1 : 0] : 0u, 0u, 0u};
          xl_u32x4 rb = {b[0], XB == 2 ? b[XB == 2 ? 1 : 0] : 0u, 0u, 0u};
          const xl_u32x2 pa = x4_bf16<XT>(ra), pb = x4_bf16<XT>(rb);
#pragma unroll
          for (int q = 0; q < 4; ++q)
            o[q][j] = (q & 1) ? ((pa[q >> 1] >> 16) | (pb[q >> 1] & 0xFFFF0000u))
                              : ((pa[q >> 1] & 0xFFFFu) | (pb[q >> 1] << 16));
        }
      }
      uint16_t* base = xl + (size_t)(so >> 2) * region * CK_PS + 8 * (so & 3);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = c + g.pw;
        if (col < g.cols)
          *reinterpret_cast<uint4*>(base + ((lo - ih0 + r) * g.cols + col) * CK_PS) =
              make_uint4(o[q][0], o[q][1], o[q][2], o[q][3]);
        if (++c == g.W) {
          c = 0;
          ++r;
        }
      }
    }
  };
  // weight run k of a lane: the 8 channels of one output channel (past the
  // last: its codes again, never stored)
  auto load_w = [&](int c0) {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int e = min(tid + 256 * k, COB * 4 - 1), co = min(co0 + (e >> 2), g.M - 1);
      const uint8_t* p = w + ((int64_t)co * g.C + c0 + 8 * (e & 3)) * T * dtype_bits(WT) / 8;
#pragma unroll
      for (int i = 0; i + 4 <= WW; i += 4) {
        const ls_u32x4u v = *reinterpret_cast<const ls_u32x4u*>(p + 4 * i);
#pragma unroll
        for (int q = 0; q < 4; ++q) wr[k][i + q] = v[q];
      }
#pragma unroll
      for (int i = WW / 4 * 4; i < WW; ++i) wr[k][i] = *reinterpret_cast<const ls_u32u*>(p + 4 * i);
    }
  };
  auto store_w = [&]() {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int e = tid + 256 * k;
      if (e >= COB * 4) continue;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        uint32_t o[2];
        ck_tap<WT, T>(wr[k], t, o);
        uint8_t* d = wl + ((t * COB + (e >> 2)) * 4 + (e & 3)) * GB;
        if constexpr (GB == 8) *reinterpret_cast<uint2*>(d) = make_uint2(o[0], o[1]);
        else *reinterpret_cast<uint32_t*>(d) = o[0];
      }
    }
  };

  load_w(0);
  load_x(0);
  for (int i = tid * 8; i < images * region * CK_PS; i += 256 * 8)
    *reinterpret_cast<uint4*>(xl + i) = make_uint4(0u, 0u, 0u, 0u);

  // staged pixel of each of the lane's tiles
  const int npix = images * g.P;
  int pb[NPX];
#pragma unroll
  for (int j = 0; j < NPX; ++j) {
    const int p = (wpx * NPX + j) * 16 + lr;
    const int im = (int)fdiv((uint32_t)p, g.fd_p), q = p - im * g.P;
    const int r = (int)fdiv((uint32_t)q, g.fd_ow), c = q - r * g.OW;
    // (a pixel outside the band reads some staged one and is never stored)
    pb[j] = p < npix && r < rows ? (im * region + r * g.sh * g.cols + c * g.sw) * CK_PS + 8 * lg
                                 : 8 * lg;
  }
  const bool live = wpx * NPX * 16 < npix;  // the wave has a pixel
  ls_f32x4 acc[NPX][NCO];
#pragma unroll
  for (int j = 0; j < NPX; ++j)
#pragma unroll
    for (int i = 0; i < NCO; ++i) acc[j][i] = ls_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  __syncthreads();  // the region is zeroed
  store_w();
  store_x();
  __syncthreads();
  const uint8_t* wf = wl + ((wco * 16 * NCO + lr) * 4 + lg) * GB;
  for (int c0 = 0; c0 < g.C; c0 += CK_C) {
    const bool more = c0 + CK_C < g.C;
    if (more) {
      load_w(c0 + CK_C);
      load_x(c0 + CK_C);
    }
    if (live) {
      // the next tap's LDS reads are on their way while a tap multiplies
      ls_bf16x8 a[2][NPX];
      uint32_t c[2][NCO][2];
      int toff = 0;
      auto read = [&](const int t, const int u) {
#pragma unroll
        for (int j = 0; j < NPX; ++j) a[u][j] = *reinterpret_cast<const ls_bf16x8*>(xl + pb[j] + toff);
#pragma unroll
        for (int i = 0; i < NCO; ++i) {
          const uint8_t* p = wf + (t * COB + 16 * i) * 4 * GB;
          if constexpr (GB == 8) {
            const uint2 v = *reinterpret_cast<const uint2*>(p);
            c[u][i][0] = v.x;
            c[u][i][1] = v.y;
          } else {
            c[u][i][0] = *reinterpret_cast<const uint32_t*>(p);
          }
        }
        if constexpr (T == 9) toff += (t % 3 == 2 ? g.cols - 2 : 1) * CK_PS;
      };
      read(0, 0);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int u = t & 1;
        if (t + 1 < T) read(t + 1, u ^ 1);
        ls_bf16x8 b[NCO];
#pragma unroll
        for (int i = 0; i < NCO; ++i) b[i] = ls_decode8<WT>(c[u][i]);
#pragma unroll
        for (int j = 0; j < NPX; ++j)
#pragma unroll
          for (int i = 0; i < NCO; ++i)
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][j], b[i], acc[j][i], 0, 0, 0);
      }
    }
    __syncthreads();
    if (more) {
      store_w();
      store_x();
      __syncthreads();
    }
  }

  // the workgroup's outputs meet in LDS half the channels at a time, then
  // leave with consecutive lanes on consecutive pixels of a channel
  const float s = product_scale(w_scale, x_scale);
  const float inv_o = epi_inv_scale(ep), z = epi_relu_factor(ep);
  constexpr int HC = COB / 2, PITCH = NPIX + 4;
  float* out = reinterpret_cast<float*>(ck_lds);
  const int64_t plane = (int64_t)g.OH * g.OW;
  uint32_t am = 0;
  // a lane keeps its pixels -- a run of 4, or one where a run would cross
  // images or miss its alignment -- and steps through the channels
  const int p = g.vec4 ? tid % (NPIX / 4) * 4 : tid % NPIX;
  const int im = (int)fdiv((uint32_t)p, g.fd_p), q0 = p - im * g.P;
  const bool in = p < npix && q0 < rows * g.OW;
  const int64_t at = (int64_t)(n0 + im) * g.M * plane + oh0 * g.OW + q0;
  for (int half = 0; half < 2; ++half) {
    if (half) __syncthreads();
    // a wave's channels 16 i + lr: its tiles of this half
#pragma unroll
    for (int i = 0; i < NCO; ++i) {
      const int row = (wco * NCO + i) * 16 - half * HC;
      if (row >= 0 && row < HC) {
#pragma unroll
        for (int j = 0; j < NPX; ++j)
          *reinterpret_cast<ls_f32x4*>(out + (row + lr) * PITCH + (wpx * NPX + j) * 16 + 4 * lg) = acc[j][i];
      }
    }
    __syncthreads();
    if (!in) continue;
    const int64_t first = (int64_t)(co0 + half * HC) * plane;
    const int last = min(HC, g.M - co0 - half * HC);
    if (g.vec4) {
      for (int r = tid / (NPIX / 4); r < last; r += 1024 / NPIX) {
        const ls_f32x4 v = *reinterpret_cast<const ls_f32x4*>(out + r * PITCH + p);
        const EpiChan k = epi_chan(ep, co0 + half * HC + r);
        float f[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f[q] = epi_value_nb(k, v[q], s, z);
          am = epi_track(am, f[q]);
        }
        epi_store4(ep.out_dtype, y, at + first + r * plane, f, inv_o);
      }
    } else {
      for (int r = tid / NPIX; r < last; r += 256 / NPIX) {
        const EpiChan k = epi_chan(ep, co0 + half * HC + r);
        const float f = epi_value_nb(k, out[r * PITCH + p], s, z);
        am = epi_track(am, f);
        epi_store(ep.out_dtype, y, at + first + r * plane, f, inv_o);
      }
    }
  }
  epi_amax_commit(ep, am);
}

// The bands of a shape for NPIX pixel slots and COB channels a workgroup, or
// false when the kernel does not take it: at most two items a lane, LDS for two
// workgroups a CU.
template <int WT, int T>
bool chunk_geometry(ChunkGeom& g, int npix_slots, int cob, int* ipt, size_t* lds) {
  if (g.C % CK_C || g.W < 4 || g.OW > npix_slots || g.N < 1) return false;
  const int64_t plane = (int64_t)g.OH * g.OW;
  if (plane <= npix_slots) {
    g.R = g.OH;
    g.G = (int)std::min<int64_t>(npix_slots / plane, g.N);
  } else {
    g.R = std::min(g.OH, npix_slots / g.OW);
    const int most = g.R, bands = (g.OH + g.R - 1) / g.R;
    g.R = (g.OH + bands - 1) / bands;
    // runs of 4 pixels stay in a band if its pixels are a multiple of 4
    while (plane % 4 == 0 && g.R * g.OW % 4 && g.R < most) ++g.R;
    g.G = 1;
  }
  g.cols = (g.OW - 1) * g.sw + g.KW;
  g.tiles_m = (g.M + cob - 1) / cob;
  const size_t wb = (size_t)T * cob * 4 * dtype_bits(WT);
  const size_t out = (size_t)cob / 2 * (npix_slots + 4) * 4;
  for (;;) {
    g.rows_in = (g.R - 1) * g.sh + g.KH;
    g.nit = (int)(((int64_t)std::min(g.rows_in, g.H) * g.W + 3) / 4);
    const int64_t items = (int64_t)g.G * 4 * g.nit;
    const size_t xb = ((size_t)g.G * g.rows_in * g.cols * CK_PS * 2 + 15) / 16 * 16;
    *lds = std::max(xb + wb, out);
    *ipt = (int)((items + 255) / 256);
    if (*ipt <= 2 && *lds <= 80 * 1024) {
      g.x_bytes = (int)xb;
      break;
    }
    if (g.G > 1) --g.G;
    else if (g.R > 1) --g.R;
    else return false;
  }
  g.bands = (g.OH + g.R - 1) / g.R;
  g.P = g.R * g.OW;
  g.groups = (g.N + g.G - 1) / g.G;
  g.vec4 = g.P % 4 == 0 && plane % 4 == 0;
  g.fd_w = fast_div((uint32_t)g.W);
  g.fd_ow = fast_div((uint32_t)g.OW);
  g.fd_p = fast_div((uint32_t)g.P);
  g.fd_nit = fast_div((uint32_t)g.nit);
  return (int64_t)g.groups * g.bands * g.tiles_m <= 0x7FFFFFFF;
}

template <int WT, int XT, int T, int NCO, int WCO, int IPT>
int chunk_launch_tile(const uint8_t* x, const float* x_scale, const uint8_t* w,
                      const float* w_scale, const Epilogue& ep, void* y, const ChunkGeom& g,
                      size_t lds, hipStream_t stream) {
  auto kern = conv2d_chunk_kernel<WT, XT, T, NCO, WCO, IPT>;
  static DeviceFlags raised;  // per instantiation
  const int rc = allow_lds(raised, reinterpret_cast<const void*>(kern), lds, 80 * 1024);
  if (rc != NOVAQ_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(g.groups * g.bands * g.tiles_m)), dim3(256), lds, stream,
                     x, x_scale, w, w_scale, ep, y, g);
  return check_launch();
}

// A shape's bands and images on one of the kernel's tiles: 0 = 32 channels x 256
// pixels, 1 = 128 x 128, 2 = 64 x 128 a workgroup.
struct ChunkPlan {
  ChunkGeom g;
  int tile, ipt;
  size_t lds;
  int64_t blocks() const { return (int64_t)g.groups * g.bands * g.tiles_m; }
};

// 64 channels x 128 pixels a workgroup; 32 x 256 for at most 32 channels; 128 x
// 128 for a strided window over many channels, whose staged region is several
// times its pixels and would be staged once per 64 channels, where that gives
// `wide_least` workgroups.
template <int WT, int T>
bool chunk_plan(const ChunkGeom& g, int wide_least, ChunkPlan& p) {
  auto tile = [&](int id, int nco, int wco) {
    p.g = g;
    p.tile = id;
    return chunk_geometry<WT, T>(p.g, 64 * (4 / wco), 16 * nco * wco, &p.ipt, &p.lds);
  };
  if (g.M <= 32) return tile(0, 2, 1);
  if (T == 9 && g.M > 64 && g.sh * g.sw > 1 && tile(1, 4, 2) && p.blocks() >= wide_least) return true;
  return tile(2, 2, 2);
}

template <int WT, int XT, int T>
int chunk_launch(const uint8_t* x, const float* x_scale, const uint8_t* w, const float* w_scale,
                 const Epilogue& ep, void* y, const ChunkPlan& p, hipStream_t stream) {
  auto go = [&](auto nco, auto wco) {
    constexpr int N = decltype(nco)::value, C = decltype(wco)::value;
    return p.ipt <= 1
               ? chunk_launch_tile<WT, XT, T, N, C, 1>(x, x_scale, w, w_scale, ep, y, p.g, p.lds, stream)
               : chunk_launch_tile<WT, XT, T, N, C, 2>(x, x_scale, w, w_scale, ep, y, p.g, p.lds, stream);
  };
  if (p.tile == 0) return go(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
  if constexpr (T == 9) {
    if (p.tile == 1) return go(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{});
  }
  return go(std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
}

}  // namespace
}  // namespace novaq
