// Kernel (a): macrocell value-range grid and majorant grid.
//
// Reference: renderer.cu:1116-1179 buildSpatialMacrocells scatters, per voxel
// (one thread each, one launch per channel), the min/max of its 3x3x3
// neighbourhood into every macrocell its widened box projects to, with CAS
// float atomics. Here the same grid is gathered instead: the host derives, per
// axis, the window of voxels whose projected boxes cover each macrocell index
// (an interval, because both projected box ends grow monotonically with the
// voxel index) and widens it by the neighbourhood. Because the window is a
// box, its min/max separates: range_pencil_kernel gives one workgroup to a
// pencil of cells along x (fixed y and z windows), reads those rows in full
// with 16-byte loads, keeps per-column min/max and reduces each cell's x
// window from LDS. Volumes whose rows are not a multiple of 16 bytes use
// range_kernel, one workgroup per (macrocell, channel) over its window in
// dword loads. No atomics, one launch for all channels.
#include "mdwt_device.hpp"
#include <algorithm>

#include "mdwt_internal.hpp"

namespace mdwt {
namespace {

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

template <int DT>
__host__ __device__ constexpr int voxel_bytes() {
  return DT == MDWT_DT_U8 ? 1 : DT == MDWT_DT_F32 ? 4 : 2;
}
// Voxel e of a little-endian dword holding 4 / voxel_bytes voxels, as
// voxel_value would convert it.
template <int DT>
__device__ __forceinline__ float word_voxel(uint32_t w, int e) {
  if constexpr (DT == MDWT_DT_U8) return float((w >> (8 * e)) & 0xffu);
  if constexpr (DT == MDWT_DT_U16) return float((w >> (16 * e)) & 0xffffu);
  if constexpr (DT == MDWT_DT_F16) {
    const uint16_t h = uint16_t(w >> (16 * e));
    return float(__builtin_bit_cast(_Float16, h));
  }
  return __uint_as_float(w);
}

template <int DT>
__global__ __launch_bounds__(256) void range_kernel(RangeParams P) {
  const int cell = blockIdx.x;
  const int ch = blockIdx.y;
  const int mx = P.mc[0], my = P.mc[1];
  const int cx = cell % mx;
  const int cy = (cell / mx) % my;
  const int cz = cell / (mx * my);
  const int* wx = P.win;
  const int* wy = P.win + 2 * P.mc[0];
  const int* wz = P.win + 2 * (P.mc[0] + P.mc[1]);
  const int x0 = wx[2 * cx], x1 = wx[2 * cx + 1];
  const int y0 = wy[2 * cy], y1 = wy[2 * cy + 1];
  const int z0 = wz[2 * cz], z1 = wz[2 * cz + 1];
  float2* out = reinterpret_cast<float2*>(P.ranges);
  if (x0 > x1 || y0 > y1 || z0 > z1) {  // no voxel covers this cell
    if (threadIdx.x == 0) out[size_t(cell) * P.channels + ch] = make_float2(1e20f, -1e20f);
    return;
  }
  const int lx = x1 - x0 + 1, ly = y1 - y0 + 1, lz = z1 - z0 + 1;
  const uint8_t* base = P.vol + size_t(ch) * P.chan_stride;
  float vmin = __int_as_float(0x7f800000), vmax = -__int_as_float(0x7f800000);
  // One row segment (lx voxels along x at fixed y, z) spans at most ndw
  // aligned dwords; gl lanes (a power of two >= ndw, at most 64) share a row
  // and rp = 256 / gl rows are read per pass, four passes' loads issued before
  // any is reduced. Rows advance by additions (iy, iz carried), no per-voxel
  // index division. A dword may hold voxels outside the window: they are
  // masked by their byte position. The channel's allocation is padded to 256
  // bytes, so the dword holding its last voxel is inside it.
  constexpr int ES = voxel_bytes<DT>();
  const int span = lx * ES;
  const int ndw = (span + 6) >> 2;
  int lg = 0;
  while ((1 << lg) < ndw && lg < 6) ++lg;
  const int gl = 1 << lg, rp = int(blockDim.x) >> lg;
  const int q = int(threadIdx.x) & (gl - 1), g = int(threadIdx.x) >> lg;
  const int nrows = ly * lz;
  const int dy = rp % ly, dz = rp / ly;
  const uint32_t nx = uint32_t(P.nx), ny = uint32_t(P.ny);
  for (int k0 = 0; k0 < ndw; k0 += gl) {
    const int k = k0 + q;
    int r = g, iy = g % ly, iz = g / ly;
    while (r < nrows) {
      uint32_t w[4];
      int s[4];
      bool ok[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        ok[u] = false;
        s[u] = 0;
        w[u] = 0u;
        if (r < nrows) {
          const size_t row = (size_t(uint32_t(z0 + iz)) * ny + uint32_t(y0 + iy)) * nx + uint32_t(x0);
          const uintptr_t lo = reinterpret_cast<uintptr_t>(base) + row * ES;
          s[u] = int(lo & 3u);
          ok[u] = k < ndw && 4 * k <= s[u] + span - 1;
          if (ok[u]) w[u] = *reinterpret_cast<const uint32_t*>((lo & ~uintptr_t(3)) + 4u * uint32_t(k));
          r += rp;
          iy += dy;
          iz += dz;
          if (iy >= ly) {
            iy -= ly;
            ++iz;
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (!ok[u]) continue;
        const int end = s[u] + span - 1;
#pragma unroll
        for (int e = 0; e < 4 / ES; ++e) {
          const int pos = 4 * k + e * ES;
          if (pos < s[u] || pos > end) continue;
          const float v = word_voxel<DT>(w[u], e);
          vmin = fminf(vmin, v);
          vmax = fmaxf(vmax, v);
        }
      }
    }
  }
  vmin = wave_min(vmin);
  vmax = wave_max(vmax);
  __shared__ float smin[4], smax[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    smin[wave] = vmin;
    smax[wave] = vmax;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float a = smin[0], b = smax[0];
    for (int w = 1; w < int(blockDim.x >> 6); ++w) {
      a = fminf(a, smin[w]);
      b = fmaxf(b, smax[w]);
    }
    // value conversion is monotone and exact on the integer types, so the
    // converted min/max equal min/max of converted voxels
    out[size_t(cell) * P.channels + ch] = make_float2(a * P.scale + P.offset, b * P.scale + P.offset);
  }
}

// Same grid, gathered per pencil: one workgroup per (cy, cz, channel) reads
// every voxel row of the pencil's y and z windows in full, as aligned 16-byte
// chunks (J chunks per lane, gl lanes per row), keeps a running min/max per x
// column in registers, merges the row slots by shuffles and the four waves in
// LDS, then reduces each cell's x window from the LDS columns. A voxel row is
// read once per (cy, cz) instead of once per cell, and each lane issues U
// chunk loads before reducing any. Requires rows of a multiple of 16 bytes
// (and at most kPencilChunks chunks); other volumes use range_kernel.
constexpr int kPencilChunks = 128;  // 16-byte chunks per row
constexpr int kPencilColumns = 2048;

template <int DT>
__device__ __forceinline__ float chunk_voxel(const uint4& c, int v) {
  const uint32_t w[4] = {c.x, c.y, c.z, c.w};
  if constexpr (DT == MDWT_DT_U8) return word_voxel<DT>(w[v >> 2], v & 3);
  if constexpr (DT == MDWT_DT_U16 || DT == MDWT_DT_F16) return word_voxel<DT>(w[v >> 1], v & 1);
  return word_voxel<DT>(w[v], 0);
}

template <int DT, int J>
__global__ __launch_bounds__(256) void range_pencil_kernel(RangeParams P) {
  constexpr int ES = voxel_bytes<DT>(), VPC = 16 / ES, U = J == 1 ? 8 : 4;
  __shared__ float cmin[kPencilColumns], cmax[kPencilColumns];
  const int cy = blockIdx.x, cz = blockIdx.y, ch = blockIdx.z;
  const int mx = P.mc[0], my = P.mc[1];
  const int* wx = P.win;
  const int* wy = P.win + 2 * P.mc[0];
  const int* wz = P.win + 2 * (P.mc[0] + P.mc[1]);
  const int y0 = wy[2 * cy], y1 = wy[2 * cy + 1];
  const int z0 = wz[2 * cz], z1 = wz[2 * cz + 1];
  float2* out = reinterpret_cast<float2*>(P.ranges) + (size_t(cz) * my + cy) * mx * P.channels + ch;
  if (y0 > y1 || z0 > z1) {  // no voxel covers any cell of the pencil
    for (int cx = threadIdx.x; cx < mx; cx += blockDim.x)
      out[size_t(cx) * P.channels] = make_float2(1e20f, -1e20f);
    return;
  }
  const int ly = y1 - y0 + 1, lz = z1 - z0 + 1, nrows = ly * lz;
  const int chunks = P.nx * ES / 16;
  int lg = 0;
  while ((1 << lg) * J < chunks && lg < 6) ++lg;
  const int gl = 1 << lg, rp = int(blockDim.x) >> lg;
  const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
  const int q = int(threadIdx.x) & (gl - 1), g = int(threadIdx.x) >> lg;
  const uint8_t* base = P.vol + size_t(ch) * P.chan_stride;
  const size_t row_bytes = size_t(P.nx) * ES;
  float vmin[J][VPC], vmax[J][VPC];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int v = 0; v < VPC; ++v) {
      vmin[j][v] = __int_as_float(0x7f800000);
      vmax[j][v] = -__int_as_float(0x7f800000);
    }
  const int dy = rp % ly, dz = rp / ly;
  int r = g, iy = g % ly, iz = g / ly;
  while (r < nrows) {
    uint4 w[U][J];
    bool ok[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ok[u] = r < nrows;
      if (ok[u]) {
        const uint8_t* row = base + (size_t(z0 + iz) * P.ny + size_t(y0 + iy)) * row_bytes;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int c = q + j * gl;
          w[u][j] = c < chunks ? *reinterpret_cast<const uint4*>(row + size_t(c) * 16) : uint4{};
        }
        r += rp;
        iy += dy;
        iz += dz;
        if (iy >= ly) {
          iy -= ly;
          ++iz;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (!ok[u]) continue;
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int v = 0; v < VPC; ++v) {
          const float x = chunk_voxel<DT>(w[u][j], v);
          vmin[j][v] = fminf(vmin[j][v], x);
          vmax[j][v] = fmaxf(vmax[j][v], x);
        }
    }
  }
  // lanes q, q + gl, ... of a wave hold the same columns (other rows)
  for (int o = gl; o < 64; o <<= 1)
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int v = 0; v < VPC; ++v) {
        vmin[j][v] = fminf(vmin[j][v], __shfl_xor(vmin[j][v], o, 64));
        vmax[j][v] = fmaxf(vmax[j][v], __shfl_xor(vmax[j][v], o, 64));
      }
  const int waves = int(blockDim.x) >> 6;
  for (int wv = 0; wv < waves; ++wv) {
    if (wave == wv && lane < gl) {
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int c = q + j * gl;
        if (c >= chunks) continue;
#pragma unroll
        for (int v = 0; v < VPC; ++v) {
          const int x = c * VPC + v;
          cmin[x] = wv == 0 ? vmin[j][v] : fminf(cmin[x], vmin[j][v]);
          cmax[x] = wv == 0 ? vmax[j][v] : fmaxf(cmax[x], vmax[j][v]);
        }
      }
    }
    __syncthreads();
  }
  // 16 lanes per cell reduce its x window from the columns
  const int sub = int(threadIdx.x) & 15;
  for (int cx0 = 0; cx0 < mx; cx0 += int(blockDim.x) >> 4) {
    const int cx = cx0 + (int(threadIdx.x) >> 4);
    const bool live = cx < mx;
    const int x0 = live ? wx[2 * cx] : 0, x1 = live ? wx[2 * cx + 1] : -1;
    float a = __int_as_float(0x7f800000), b = -__int_as_float(0x7f800000);
    for (int x = x0 + sub; x <= x1; x += 16) {
      a = fminf(a, cmin[x]);
      b = fmaxf(b, cmax[x]);
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) {
      a = fminf(a, __shfl_xor(a, o, 64));
      b = fmaxf(b, __shfl_xor(b, o, 64));
    }
    if (live && sub == 0)
      out[size_t(cx) * P.channels] = x0 > x1 ? make_float2(1e20f, -1e20f)
                                             : make_float2(a * P.scale + P.offset,
                                                           b * P.scale + P.offset);
  }
}

// Majorants. A cell's majorant in a channel is the largest of the opacities at
// the texels its value range covers, so the opacity of every texel is computed
// once per workgroup into LDS, and a maximum over texels does not depend on the
// order. (With a lookup and a division per texel and one lane per cell, 55 k cells
// of three channels took 42 us and 512 cells of four 121 us.)
//
// SPREAD: a group of kMajLanes lanes per entry takes its texels side by side.
// Otherwise a lane per entry: it takes a short range alone, and its group takes the
// longer ones together, one after another. A rebuild (the whole call) of one slider's
// change, smooth data: 64^3 cells of four channels, 64 texels: 91 us spread, 24 with a
// lane each (33 with one lane and a lookup per texel); 128^3 cells, 16 texels: 572 and
// 58 us (76); 38^3 cells, 256 texels: 37 and 46 us (53); 24^3 cells, 2048 texels, one
// channel of noise: 39 and 118 us (430).
constexpr int kMajLanes = 16;
// A lane each wins from about 64 k entries on; below, with long tables, the entries
// alone leave the chip idle. The shorter the table, the less there is to spread: with
// 64 texels the two meet between 14 and 33 k entries (four channels' sums: 22.5 us
// spread against 25.5 at 13.8 k, 27.1 against 21.9 at 32.8 k), with 16 or fewer below 14 k
// (18.0 against 17.2).
inline int spread_entries(int texels) { return texels <= 32 ? 4096 : (texels <= 128 ? 16384 : 65536); }

// maximum over the kMajLanes lanes of a group
__device__ __forceinline__ float group_max(float m) {
#pragma unroll
  for (int o = kMajLanes / 2; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  return m;
}
// maximum (at least 0) of table[at + i], i = i0 .. i1: SPREAD for the group's one
// interval, otherwise for every lane's own (all lanes of the group call it)
template <bool SPREAD>
__device__ __forceinline__ float interval_max(const float* table, int at, int i0, int i1) {
  const int sub = threadIdx.x % kMajLanes, first = (threadIdx.x & 63) - sub;
  float m = 0.f;
  if (SPREAD) {
    for (int i = i0 + sub; i <= i1; i += kMajLanes) m = fmaxf(m, table[at + i]);
    return group_max(m);
  }
  const bool wide = i1 - i0 >= kMajLanes;
  if (!wide)
    for (int i = i0; i <= i1; ++i) m = fmaxf(m, table[at + i]);
  uint32_t todo = uint32_t(__ballot(wide) >> first) & ((1u << kMajLanes) - 1u);
  while (todo) {  // the same for the lanes of a group
    const int l = __builtin_ctz(todo);
    todo &= todo - 1u;
    const int j0 = __shfl(i0, first + l, 64), j1 = __shfl(i1, first + l, 64), t = __shfl(at, first + l, 64);
    float x = 0.f;
    for (int i = j0 + sub; i <= j1; i += kMajLanes) x = fmaxf(x, table[t + i]);
    x = group_max(x);
    if (sub == l) m = x;
  }
  return m;
}

// Per-channel majorant of one cell, renderer.cu:159-203 (the texel-interval
// max plus the two extra lerp lookups at addr + 0.5). at_texel[at + i]: the channel's
// opacity looked up at texel i, (i + 0.5) / n; 0 without any (an empty range).
template <bool SPREAD>
__device__ __forceinline__ float channel_majorant(const float* at_texel, int at, const float4* tab, int n,
                                                  float os, float xlo, float xhi, float vlo, float vhi,
                                                  float mn, float mx, bool any) {
  const float remappedMin1 = (mn - vlo) / (vhi - vlo);
  const float remappedMin = (remappedMin1 - xlo) / (xhi - xlo);
  const float remappedMax1 = (mx - vlo) / (vhi - vlo);
  const float remappedMax = (remappedMax1 - xlo) / (xhi - xlo);
  const float addr1 = remappedMin * float(n);
  const float addr2 = remappedMax * float(n);
  const int addrMin = clamp_index(fminf(floorf(addr1), floorf(addr2)), n);
  const int addrMax = clamp_index(fmaxf(ceilf(addr1), ceilf(addr2)), n);
  float m = interval_max<SPREAD>(at_texel, at, addrMin, any ? addrMax : addrMin - 1);
  if (!any) return 0.f;
  float d = tf_lerp_alpha(tab, n, (addr1 + 0.5f) / float(n)) * os;
  m = fmaxf(m, d);
  d = tf_lerp_alpha(tab, n, (addr2 + 0.5f) / float(n)) * os;
  m = fmaxf(m, d);
  return m;
}

// An option beside renderer.cu:159-203, whose majorant can fall below the
// opacities a lookup interpolates by up to half a texel of lerp: the largest
// opacity of every texel that a lookup of a value in [mn, mx] reads. The
// lookup interval is widened by 2^-12 (1 + |r|) on each side, which covers the
// render's remap by reciprocals against the divisions here, and the maximum
// is scaled by 1 + 2^-20 for the lerp's rounding. A lookup at u reads
// texels floor(u n - 0.5) and the next one, clamped to the table. texel[at + i]: the
// channel's stored opacity.
template <bool SPREAD>
__device__ __forceinline__ float channel_majorant_conservative(const float* texel, int at, int n, float os,
                                                               float xlo, float xhi, float vlo,
                                                               float vhi, float mn, float mx, bool any) {
  const float r1 = ((mn - vlo) / (vhi - vlo) - xlo) / (xhi - xlo);
  const float r2 = ((mx - vlo) / (vhi - vlo) - xlo) / (xhi - xlo);
  const float a = fminf(r1, r2), b = fmaxf(r1, r2);
  const float lo = a - 0x1p-12f * (1.0f + fabsf(a)), hi = b + 0x1p-12f * (1.0f + fabsf(b));
  const int i0 = clamp_index(floorf(lo * float(n) - 0.5f), n);
  const int i1 = clamp_index_plus1(floorf(hi * float(n) - 0.5f), n);
  const float m = interval_max<SPREAD>(texel, at, i0, any ? i1 : i0 - 1);
  return any ? m * os * (1.0f + 0x1p-20f) : 0.f;
}

// renderer.cu:206-274: modes 0-2 keep one majorant per (cell, channel)
// (renderer.cu:159-203), modes 3-9 their sum per cell (renderer.cu:111-157).
// A group of kMajLanes lanes (SPREAD) or a lane per entry; workgroups stride over
// the entries.
template <bool SPREAD>
__global__ __launch_bounds__(256) void majorant_kernel(MajorantParams P) {
  extern __shared__ float s_texel[];  // [channel][stride]
  const int C = P.channels, stride = P.tf.stride;
  const float4* tab = reinterpret_cast<const float4*>(P.tf.tab);
  const float2* rg = reinterpret_cast<const float2*>(P.ranges);
  for (int k = threadIdx.x; k < C * stride; k += blockDim.x) {
    const int c = k / stride, i = k - c * stride, n = P.tf.n[c];
    float v = 0.f;
    if (i < n)
      v = P.conservative ? tab[k].w
                         : tf_lerp_alpha(tab + size_t(c) * stride, n, (float(i) + 0.5f) / float(n)) *
                               P.tf.opacity[c];
    s_texel[k] = v;
  }
  __syncthreads();
  auto majorant = [&](const float2 r, int c, bool any) {
    any = any && !(r.y < r.x);
    const int at = c * stride;
    return P.conservative
               ? channel_majorant_conservative<SPREAD>(s_texel, at, P.tf.n[c], P.tf.opacity[c], P.tf.xf_lo[c],
                                                       P.tf.xf_hi[c], P.tf.dom_lo[c], P.tf.dom_hi[c], r.x, r.y, any)
               : channel_majorant<SPREAD>(s_texel, at, tab + size_t(c) * stride, P.tf.n[c], P.tf.opacity[c],
                                          P.tf.xf_lo[c], P.tf.xf_hi[c], P.tf.dom_lo[c], P.tf.dom_hi[c], r.x, r.y,
                                          any);
  };
  const int entries = P.mode <= 2 ? P.n_cells * C : P.n_cells;
  constexpr int kLanes = SPREAD ? kMajLanes : 1, kPer = 256 / kLanes;
  const int own = int(threadIdx.x) / kLanes;
  for (int i0 = int(blockIdx.x) * kPer; i0 < entries; i0 += int(gridDim.x) * kPer) {
    const bool any = i0 + own < entries;
    const int i = any ? i0 + own : 0;
    float m = 0.f;
    if (P.mode <= 2) {
      m = majorant(rg[i], i % C, any);
    } else {
      for (int c = 0; c < C; ++c) m += majorant(rg[size_t(i) * C + c], c, any);
    }
    if (any && threadIdx.x % kLanes == 0) P.maj[i] = m;
  }
}

// Cost-sorted block order (longest processing time first): the nb blocks of
// `order` by the summed wall-clock ticks of their wpb waves, heaviest first, in
// place (tmp: nb entries). Workgroup i runs on XCD i % 8, so the list is dealt
// round-robin over the XCDs and the slowest blocks start first instead of
// trailing at the end of the frame. One workgroup, a counting sort into 1024
// classes of equal width (the order inside a class does not matter): the ticks
// used to go to the host and the order back, 85 us of a 234 us one-frame call at
// 4096 blocks.
//
// Up to kSortKeep blocks per thread (a 1024^2 frame of 16x16 blocks) the costs and
// the order are read once, kept in registers and written straight to their
// places; larger frames read the ticks again for each phase and go through tmp.
// The kernel is a chain of latencies, on the path of every first frame of an
// accumulation: 17.0 -> 5.9 us at 4096 blocks, 10.0 -> 4.5 us at 1938.
constexpr int kSortThreads = 1024;
constexpr int kSortKeep = 4;
__global__ __launch_bounds__(kSortThreads) void cost_order_kernel(uint32_t* order, const uint32_t* ticks,
                                                                  uint32_t* tmp, int nb, int wpb) {
  __shared__ uint32_t s_cnt[kSortThreads];
  __shared__ uint32_t s_wave[kSortThreads / 64];
  __shared__ uint32_t s_max;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  auto cost = [&](int b) -> uint32_t {
    uint32_t c = 0;
    if (wpb == 4) {  // one load instead of four in a loop
      const uint4 q = reinterpret_cast<const uint4*>(ticks)[b];
      return min(q.x, 0x3fffffffu) + min(q.y, 0x3fffffffu) + min(q.z, 0x3fffffffu) + min(q.w, 0x3fffffffu);
    }
    for (int w = 0; w < wpb; ++w) c += min(ticks[size_t(wpb) * b + w], 0x3fffffffu);
    return c;
  };
  const bool keep = nb <= kSortKeep * kSortThreads;
  uint32_t kc[kSortKeep], ko[kSortKeep];
#pragma unroll
  for (int k = 0; k < kSortKeep; ++k) {
    const int b = t + k * kSortThreads;
    const bool in = keep && b < nb;
    kc[k] = in ? cost(b) : 0u;
    ko[k] = in ? order[b] : 0u;
  }
  // each(b, cost, order) over this thread's blocks
  auto each = [&](auto&& use) {
    if (keep) {
#pragma unroll
      for (int k = 0; k < kSortKeep; ++k)
        if (t + k * kSortThreads < nb) use(kc[k], ko[k]);
    } else {
      for (int b = t; b < nb; b += kSortThreads) use(cost(b), order[b]);
    }
  };
  // the order's words have arrived before any thread writes its own
#pragma unroll
  for (int k = 0; k < kSortKeep; ++k) asm volatile("" ::"v"(ko[k]));
  if (t == 0) s_max = 1u;
  s_cnt[t] = 0u;
  __syncthreads();
  uint32_t top = 0u;
  each([&](uint32_t c, uint32_t) { top = max(top, c); });
  for (int o = 32; o > 0; o >>= 1) top = max(top, uint32_t(__shfl_xor(int(top), o, 64)));
  if (lane == 0) atomicMax(&s_max, top);
  __syncthreads();
  const float scale = float(kSortThreads - 1) / float(s_max);
  auto cls = [&](uint32_t c) {  // class 0: the heaviest
    return kSortThreads - 1 - min(kSortThreads - 1, int(float(c) * scale));
  };
  each([&](uint32_t c, uint32_t) { atomicAdd(&s_cnt[cls(c)], 1u); });
  __syncthreads();
  // the start of every class: prefix sums within a wave, then over the waves
  const uint32_t own = s_cnt[t];
  uint32_t sum = own;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t v = uint32_t(__shfl_up(int(sum), o, 64));
    if (lane >= o) sum += v;
  }
  if (lane == 63) s_wave[wave] = sum;
  __syncthreads();
  uint32_t before = lane < wave ? s_wave[lane] : 0u;  // 16 waves
  for (int o = 8; o > 0; o >>= 1) before += uint32_t(__shfl_xor(int(before), o, 64));
  s_cnt[t] = uint32_t(__shfl(int(before), 0, 64)) + sum - own;
  __syncthreads();
  uint32_t* out = keep ? order : tmp;  // kept: every thread has read its part of order
  each([&](uint32_t c, uint32_t o) { out[atomicAdd(&s_cnt[cls(c)], 1u)] = o; });
  if (keep) return;
  __threadfence_block();
  __syncthreads();
  for (int b = t; b < nb; b += kSortThreads) order[b] = tmp[b];
}

// Brick copy of the volume (the samplers' layout, VolumeParams): output
// voxel o of a channel is voxel (o & 3, (o >> 2) & 3, o >> 4) of brick
// o >> 6 (bricks x fastest); voxels past the volume's edge are zero (the
// samplers clamp their indices, so they are never read). One thread per
// output voxel, grid (bricks * 64 / 256, channels).
template <typename T>
__global__ __launch_bounds__(256) void brick_kernel(const uint8_t* __restrict__ vol, uint64_t chan_stride,
                                                    int nx, int ny, int nz, int nbx, int nby,
                                                    uint64_t per, uint8_t* __restrict__ bricks,
                                                    uint64_t brick_stride) {
  const uint64_t o = uint64_t(blockIdx.x) * 256u + threadIdx.x;
  if (o >= per) return;
  const uint32_t b = uint32_t(o >> 6), w = uint32_t(o & 63u);
  const uint32_t bx = b % uint32_t(nbx), r = b / uint32_t(nbx);
  const uint32_t by = r % uint32_t(nby), bz = r / uint32_t(nby);
  const uint32_t x = bx * 4u + (w & 3u), y = by * 4u + ((w >> 2) & 3u), z = bz * 4u + (w >> 4);
  const T* src = reinterpret_cast<const T*>(vol + size_t(blockIdx.y) * chan_stride);
  T* dst = reinterpret_cast<T*>(bricks + size_t(blockIdx.y) * brick_stride);
  dst[o] = (x < uint32_t(nx) && y < uint32_t(ny) && z < uint32_t(nz))
               ? src[(size_t(z) * uint32_t(ny) + y) * uint32_t(nx) + x]
               : T(0);
}

// Joint copy (VolumeParams::joint): output voxel o of group blockIdx.y holds
// channels 4 g .. 4 g + 3 of brick_kernel's voxel o side by side (zero past the
// last channel). One thread per output voxel: the reads of a channel are the
// brick copy's, the write is one 4-, 8- or 16-byte store.
template <typename T>
__global__ __launch_bounds__(256) void joint_kernel(const uint8_t* __restrict__ vol, uint64_t chan_stride,
                                                    int channels, int nx, int ny, int nz, int nbx,
                                                    int nby, uint64_t per, uint8_t* __restrict__ joint,
                                                    uint64_t joint_stride) {
  struct alignas(4 * sizeof(T)) T4 {
    T v[4];
  };
  const uint64_t o = uint64_t(blockIdx.x) * 256u + threadIdx.x;
  if (o >= per) return;
  const uint32_t b = uint32_t(o >> 6), w = uint32_t(o & 63u);
  const uint32_t bx = b % uint32_t(nbx), r = b / uint32_t(nbx);
  const uint32_t by = r % uint32_t(nby), bz = r / uint32_t(nby);
  const uint32_t x = bx * 4u + (w & 3u), y = by * 4u + ((w >> 2) & 3u), z = bz * 4u + (w >> 4);
  const bool in = x < uint32_t(nx) && y < uint32_t(ny) && z < uint32_t(nz);
  const size_t at = in ? (size_t(z) * uint32_t(ny) + y) * uint32_t(nx) + x : 0;
  T4 q;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = 4 * int(blockIdx.y) + k;
    q.v[k] = in && c < channels ? reinterpret_cast<const T*>(vol + size_t(c) * chan_stride)[at] : T(0);
  }
  reinterpret_cast<T4*>(joint + size_t(blockIdx.y) * joint_stride)[o] = q;
}

template <int DT>
void launch_pencils(const RangeParams& p, hipStream_t s) {
  const dim3 grid(unsigned(p.mc[1]), unsigned(p.mc[2]), unsigned(p.channels));
  if (p.nx * voxel_bytes<DT>() <= 64 * 16)
    hipLaunchKernelGGL((range_pencil_kernel<DT, 1>), grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((range_pencil_kernel<DT, 2>), grid, dim3(256), 0, s, p);
}

int dtype_bytes(int dtype) { return dtype == MDWT_DT_U8 ? 1 : dtype == MDWT_DT_F32 ? 4 : 2; }

}  // namespace

hipError_t launch_ranges(const RangeParams& p, int dtype, hipStream_t s) {
  const int row = p.nx * dtype_bytes(dtype);
  if (row % 16 == 0 && row / 16 <= kPencilChunks) {
    switch (dtype) {
      case MDWT_DT_U8: launch_pencils<MDWT_DT_U8>(p, s); break;
      case MDWT_DT_U16: launch_pencils<MDWT_DT_U16>(p, s); break;
      case MDWT_DT_F16: launch_pencils<MDWT_DT_F16>(p, s); break;
      default: launch_pencils<MDWT_DT_F32>(p, s); break;
    }
    return hipGetLastError();
  }
  const int n_cells = p.mc[0] * p.mc[1] * p.mc[2];
  const dim3 grid(unsigned(n_cells), unsigned(p.channels));
  switch (dtype) {
    case MDWT_DT_U8: hipLaunchKernelGGL(range_kernel<MDWT_DT_U8>, grid, dim3(256), 0, s, p); break;
    case MDWT_DT_U16: hipLaunchKernelGGL(range_kernel<MDWT_DT_U16>, grid, dim3(256), 0, s, p); break;
    case MDWT_DT_F16: hipLaunchKernelGGL(range_kernel<MDWT_DT_F16>, grid, dim3(256), 0, s, p); break;
    default: hipLaunchKernelGGL(range_kernel<MDWT_DT_F32>, grid, dim3(256), 0, s, p); break;
  }
  return hipGetLastError();
}

hipError_t launch_bricks(const VolumeParams& v, int dtype, hipStream_t s) {
  const uint64_t per = uint64_t(v.nbx) * uint64_t(v.nby) * uint64_t((v.nz + 3) / 4) * 64u;
  const dim3 grid(unsigned((per + 255) / 256), unsigned(v.channels));
  switch (dtype_bytes(dtype)) {
    case 1:
      hipLaunchKernelGGL(brick_kernel<uint8_t>, grid, dim3(256), 0, s, v.vol, v.chan_stride, v.nx, v.ny,
                         v.nz, v.nbx, v.nby, per, const_cast<uint8_t*>(v.bricks), v.brick_stride);
      break;
    case 2:
      hipLaunchKernelGGL(brick_kernel<uint16_t>, grid, dim3(256), 0, s, v.vol, v.chan_stride, v.nx, v.ny,
                         v.nz, v.nbx, v.nby, per, const_cast<uint8_t*>(v.bricks), v.brick_stride);
      break;
    default:
      hipLaunchKernelGGL(brick_kernel<uint32_t>, grid, dim3(256), 0, s, v.vol, v.chan_stride, v.nx, v.ny,
                         v.nz, v.nbx, v.nby, per, const_cast<uint8_t*>(v.bricks), v.brick_stride);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_joint(const VolumeParams& v, int dtype, hipStream_t s) {
  const uint64_t per = uint64_t(v.nbx) * uint64_t(v.nby) * uint64_t((v.nz + 3) / 4) * 64u;
  const dim3 grid(unsigned((per + 255) / 256), unsigned((v.channels + 3) / 4));
  uint8_t* out = const_cast<uint8_t*>(v.joint);
  switch (dtype_bytes(dtype)) {
    case 1:
      hipLaunchKernelGGL(joint_kernel<uint8_t>, grid, dim3(256), 0, s, v.vol, v.chan_stride, v.channels,
                         v.nx, v.ny, v.nz, v.nbx, v.nby, per, out, v.joint_stride);
      break;
    case 2:
      hipLaunchKernelGGL(joint_kernel<uint16_t>, grid, dim3(256), 0, s, v.vol, v.chan_stride, v.channels,
                         v.nx, v.ny, v.nz, v.nbx, v.nby, per, out, v.joint_stride);
      break;
    default:
      hipLaunchKernelGGL(joint_kernel<uint32_t>, grid, dim3(256), 0, s, v.vol, v.chan_stride, v.channels,
                         v.nx, v.ny, v.nz, v.nbx, v.nby, per, out, v.joint_stride);
      break;
  }
  return hipGetLastError();
}

hipError_t launch_majorants(const MajorantParams& p, hipStream_t s) {
  const int work = p.mode <= 2 ? p.n_cells * p.channels : p.n_cells;
  const bool spread = work <= spread_entries(p.tf.stride);
  const int per = spread ? 256 / kMajLanes : 256, blocks = std::min((work + per - 1) / per, 2048);
  // at most kMaxTexelsLds floats (40 KiB)
  const size_t lds = size_t(p.channels) * size_t(p.tf.stride) * sizeof(float);
  hipLaunchKernelGGL(spread ? majorant_kernel<true> : majorant_kernel<false>, dim3(unsigned(blocks)), dim3(256), lds,
                     s, p);
  return hipGetLastError();
}

hipError_t launch_cost_order(uint32_t* order, const uint32_t* ticks, uint32_t* tmp, int nb, int wpb,
                             hipStream_t s) {
  hipLaunchKernelGGL(cost_order_kernel, dim3(1), dim3(kSortThreads), 0, s, order, ticks, tmp, nb, wpb);
  return hipGetLastError();
}

}  // namespace mdwt
