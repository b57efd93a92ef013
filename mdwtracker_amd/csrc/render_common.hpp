// Shared device pieces of the frame kernels: per-channel transfer functions
// in LDS, volume sampling, work counters and the block schedule.
#pragma once
#include "mdwt_device.hpp"

namespace mdwt {

// Per-channel transfer-function parameters in LDS: value domain [dlo, dhi],
// TF range start xlo, the correctly rounded reciprocals of the domain width
// (idw) and of the TF range width (ixw), opacity scale, texel count and
// texel offset.
struct ChanTf {
  float dlo, dhi, xlo, ixw, os;
  int n;
  int off;  // texel offset in LDS
  float idw;
};

struct Counts {
  uint32_t samples, visits, rejections, rays;
};

struct HitRec {
  bool missed;
  float r, g, b;
  float a;  // transparency: 1 for a Woodcock hit, the composited alpha for the marchers
  float tHit;
  int channel;
};

template <int DT>
struct Ctx {
  const uint8_t* bricks;
  uint64_t brick_stride;
  const uint8_t* joint;
  uint64_t joint_stride;
  bool bricks32;       // every channel's bricks within 4 GiB
  uint32_t nbx, nbxy;  // bricks per row and per slab (both below 2^24)
  int nx, ny, nz;
  float scale, offset;
  const float4* tf;    // LDS
  const ChanTf* chtf;  // LDS
  const float* maj;
  int C;
  int mx, my, mz;
  float dt;

  __device__ __forceinline__ void init(const RenderParams& P, const float4* tf_lds,
                                       const ChanTf* ch_lds) {
    bricks = P.vol.bricks;
    brick_stride = P.vol.brick_stride;
    bricks32 = brick_stride * uint64_t(P.vol.channels) <= 0xffffffffull;
    joint = P.vol.joint;
    joint_stride = P.vol.joint_stride;
    nbx = uint32_t(P.vol.nbx);
    nbxy = nbx * uint32_t(P.vol.nby);
    nx = P.vol.nx;
    ny = P.vol.ny;
    nz = P.vol.nz;
    scale = P.vol.scale;
    offset = P.vol.offset;
    tf = tf_lds;
    chtf = ch_lds;
    maj = P.maj;
    C = P.vol.channels;
    mx = P.mc[0];
    my = P.mc[1];
    mz = P.mc[2];
    dt = P.dt;
  }

  // sampleVolumeTexture (deviceCode.cu:122-132): NaN outside [0,1]^3, else
  // clamp-to-edge trilinear at texel coordinate p*N - 0.5. In two parts, so
  // that a caller can do other work while the voxels are on their way:
  // corners() issues the eight loads (indices are clamped, so they are in
  // bounds for every p, NaN included), trilinear() waits for them.
  static constexpr uint32_t kBytes = DT == MDWT_DT_U8 ? 1u : (DT == MDWT_DT_F32 ? 4u : 2u);
  struct Corners {
    uint32_t b000, b100, b010, b110, b001, b101, b011, b111;  // stored bits
    float fx, fy, fz;
    bool inside;
    // the point up to which other work may run while the loads are in flight
    __device__ __forceinline__ void arrived() {
      asm volatile("" : "+v"(b000), "+v"(b100), "+v"(b010), "+v"(b110), "+v"(b001), "+v"(b101),
                        "+v"(b011), "+v"(b111));
    }
  };
  // The footprint of a position: the voxel indices of its eight corners
  // (x fastest), the lerp weights, and whether it is in the unit cube.
  struct Foot {
    uint32_t i[8];
    float fx, fy, fz;
    bool inside;
  };
  __device__ __forceinline__ Foot foot(V3 p) const {
    Foot k;
    k.inside = !(p.x < 0.0f || p.x > 1.0f || p.y < 0.0f || p.y > 1.0f || p.z < 0.0f || p.z > 1.0f);
    const float x = p.x * float(nx) - 0.5f;
    const float y = p.y * float(ny) - 0.5f;
    const float z = p.z * float(nz) - 0.5f;
    const float flx = floorf(x), fly = floorf(y), flz = floorf(z);
    k.fx = x - flx;
    k.fy = y - fly;
    k.fz = z - flz;
    int x0, x1, y0, y1, z0, z1;
    clamp_pair(flx, nx, x0, x1);
    clamp_pair(fly, ny, y0, y1);
    clamp_pair(flz, nz, z0, z1);
    // the voxels are read from the 4 x 4 x 4 brick copies: index = X(x) +
    // Y(y) + Z(z) (a trilinear footprint touches about 1.8 cache lines
    // instead of 4 in the planar layout; 3.5% faster at -m 2 on 4 x 256^3 u8)
    const uint32_t ax0 = (uint32_t(x0 >> 2) << 6) | (x0 & 3), ax1 = (uint32_t(x1 >> 2) << 6) | (x1 & 3);
    // brick coordinates and the bricks per row / slab are below 2^24 (checked
    // when the volume is set)
    const uint32_t ay0 = (mul_u24(y0 >> 2, nbx) << 6) | ((y0 & 3) << 2);
    const uint32_t ay1 = (mul_u24(y1 >> 2, nbx) << 6) | ((y1 & 3) << 2);
    const uint32_t az0 = (mul_u24(z0 >> 2, nbxy) << 6) | ((z0 & 3) << 4);
    const uint32_t az1 = (mul_u24(z1 >> 2, nbxy) << 6) | ((z1 & 3) << 4);
    const uint32_t r00 = ay0 + az0, r10 = ay1 + az0, r01 = ay0 + az1, r11 = ay1 + az1;
    k.i[0] = r00 + ax0;
    k.i[1] = r00 + ax1;
    k.i[2] = r10 + ax0;
    k.i[3] = r10 + ax1;
    k.i[4] = r01 + ax0;
    k.i[5] = r01 + ax1;
    k.i[6] = r11 + ax0;
    k.i[7] = r11 + ax1;
    return k;
  }
  __device__ __forceinline__ Corners corners(V3 p, int c) const {
    const Foot f = foot(p);
    Corners k;
    k.inside = f.inside;
    k.fx = f.fx;
    k.fy = f.fy;
    k.fz = f.fz;
    if (bricks32) {
      // byte offsets from the array's uniform base in 32 bits (channel bases
      // differ between lanes): no 64-bit address per voxel
      const uint32_t at = uint32_t(c) * uint32_t(brick_stride);
      k.b000 = fetch_bits_at<DT>(bricks, at + f.i[0] * kBytes);
      k.b100 = fetch_bits_at<DT>(bricks, at + f.i[1] * kBytes);
      k.b010 = fetch_bits_at<DT>(bricks, at + f.i[2] * kBytes);
      k.b110 = fetch_bits_at<DT>(bricks, at + f.i[3] * kBytes);
      k.b001 = fetch_bits_at<DT>(bricks, at + f.i[4] * kBytes);
      k.b101 = fetch_bits_at<DT>(bricks, at + f.i[5] * kBytes);
      k.b011 = fetch_bits_at<DT>(bricks, at + f.i[6] * kBytes);
      k.b111 = fetch_bits_at<DT>(bricks, at + f.i[7] * kBytes);
    } else {
      const uint8_t* base = bricks + size_t(c) * brick_stride;
      k.b000 = fetch_bits<DT>(base, f.i[0]);
      k.b100 = fetch_bits<DT>(base, f.i[1]);
      k.b010 = fetch_bits<DT>(base, f.i[2]);
      k.b110 = fetch_bits<DT>(base, f.i[3]);
      k.b001 = fetch_bits<DT>(base, f.i[4]);
      k.b101 = fetch_bits<DT>(base, f.i[5]);
      k.b011 = fetch_bits<DT>(base, f.i[6]);
      k.b111 = fetch_bits<DT>(base, f.i[7]);
      k.arrived();  // (keeps the compiler from merging the two branches' loads again)
    }
    return k;
  }
  __device__ __forceinline__ float lerp8(const float v[8], float fx, float fy, float fz,
                                         bool inside) const {
    const float c00 = v[0] + fx * (v[1] - v[0]);
    const float c10 = v[2] + fx * (v[3] - v[2]);
    const float c01 = v[4] + fx * (v[5] - v[4]);
    const float c11 = v[6] + fx * (v[7] - v[6]);
    const float c0 = c00 + fy * (c10 - c00);
    const float c1 = c01 + fy * (c11 - c01);
    const float r = c0 + fz * (c1 - c0);
    return inside ? r * scale + offset : qnan();
  }
  __device__ __forceinline__ float trilinear(Corners k) const {
    // All eight loads in flight before the first value is used: left to itself
    // the scheduler saves address registers by issuing one load, waiting for it
    // and reusing its address pair, in some instances and not in others.
    asm("" : "+v"(k.b000), "+v"(k.b100), "+v"(k.b010), "+v"(k.b110), "+v"(k.b001), "+v"(k.b101),
             "+v"(k.b011), "+v"(k.b111));
    const float v[8] = {voxel_value<DT>(k.b000), voxel_value<DT>(k.b100), voxel_value<DT>(k.b010),
                        voxel_value<DT>(k.b110), voxel_value<DT>(k.b001), voxel_value<DT>(k.b101),
                        voxel_value<DT>(k.b011), voxel_value<DT>(k.b111)};
    return lerp8(v, k.fx, k.fy, k.fz, k.inside);
  }

  // Every channel at one position, in channel order. With the joint copy a
  // corner's four channels are one load (4, 8 or 16 bytes), so a group of four
  // takes eight loads and addresses instead of 32: the ray marchers, bound by
  // VALU issue, went from 805 to 619 us a frame (-m 8, 640 x 480, 4 x 128^3 u8)
  // with the next step's loads under this step's blend, and -m 3 / 4 / 5 from
  // 73 / 79 / 79 to 38 / 39 / 38 us (half of it from several frames per launch).
  // Without the copy (one channel, or no memory for it) each channel is loaded
  // by itself. The first loads
  // are issued by all_channels(), the rest as each() gets there.
  static constexpr int kWords = DT == MDWT_DT_U8 ? 1 : (DT == MDWT_DT_F32 ? 4 : 2);
  struct AllChannels {
    Foot f;
    uint32_t w[8][kWords];
    __device__ __forceinline__ void arrived() {
#pragma unroll
      for (int j = 0; j < kWords; ++j)
        asm volatile("" : "+v"(w[0][j]), "+v"(w[1][j]), "+v"(w[2][j]), "+v"(w[3][j]),
                          "+v"(w[4][j]), "+v"(w[5][j]), "+v"(w[6][j]), "+v"(w[7][j]));
    }
  };
  // a voxel of a group of the joint copy
  template <class Offset>
  static __device__ __forceinline__ void load_group(uint32_t (&w)[kWords], const uint8_t* base, Offset at) {
    if constexpr (kWords == 1) {
      w[0] = *reinterpret_cast<const uint32_t*>(base + at);
    } else if constexpr (kWords == 2) {
      const uint2 v = *reinterpret_cast<const uint2*>(base + at);
      w[0] = v.x;
      w[1] = v.y;
    } else {
      const uint4 v = *reinterpret_cast<const uint4*>(base + at);
      w[0] = v.x;
      w[1] = v.y;
      w[2] = v.z;
      w[3] = v.w;
    }
  }
  __device__ __forceinline__ void load_channels(AllChannels& a, int c0) const {
    if (joint) {
      const uint8_t* base = joint + size_t(c0 >> 2) * joint_stride;
      if (joint_stride <= 0xffffffffull) {  // 32-bit byte offsets, as corners()
#pragma unroll
        for (int i = 0; i < 8; ++i) load_group(a.w[i], base, a.f.i[i] * (4u * kBytes));
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) load_group(a.w[i], base, uint64_t(a.f.i[i]) * (4u * kBytes));
        a.arrived();
      }
    } else {
      const uint8_t* base = bricks + size_t(c0) * brick_stride;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        a.w[i][0] = fetch_bits<DT>(base, a.f.i[i]);
#pragma unroll
        for (int j = 1; j < kWords; ++j) a.w[i][j] = 0u;
      }
    }
  }
  __device__ __forceinline__ AllChannels all_channels(V3 p) const {
    AllChannels a;
    a.f = foot(p);
    load_channels(a, 0);
    return a;
  }
  // use(c, value) for channel 0, 1, ... until it returns false (value: NaN
  // outside the unit cube)
  template <class Use>
  __device__ __forceinline__ void each(AllChannels& a, const Use& use) const {
    const int step = joint ? 4 : 1;
    for (int c0 = 0;;) {
      a.arrived();
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (k >= step || c0 + k >= C) break;
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t bits = DT == MDWT_DT_U8    ? (a.w[i][0] >> (8 * k)) & 0xffu
                                : DT == MDWT_DT_F32 ? a.w[i][k]
                                                    : (a.w[i][k >> 1] >> (16 * (k & 1))) & 0xffffu;
          v[i] = voxel_value<DT>(bits);
        }
        if (!use(c0 + k, lerp8(v, a.f.fx, a.f.fy, a.f.fz, a.f.inside))) return;
      }
      c0 += step;
      if (c0 >= C) return;
      load_channels(a, c0);
    }
  }

  // The value of one channel that is the same for the whole wave (NaN outside the
  // unit cube), as in the thread-per-pixel kernels' channel loops: the channel's
  // base is scalar. corners(), whose offsets count from the array's base, costs
  // them an addition per voxel, a second address path and its registers (-m 9,
  // 300 x 200, 128^3 u8: 640 -> 720 us on four channels; shaded batched views in
  // launch form 2 fell from three waves per SIMD to two). All eight loads are
  // issued before the first value is used (see trilinear).
  __device__ __forceinline__ float sample(V3 p, int c) const {
    if (p.x < 0.0f || p.x > 1.0f || p.y < 0.0f || p.y > 1.0f || p.z < 0.0f || p.z > 1.0f)
      return qnan();
    const Foot f = foot(p);
    const uint8_t* base = bricks + size_t(c) * brick_stride;
    uint32_t w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = fetch_bits<DT>(base, f.i[i]);
    asm("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(w[4]), "+v"(w[5]), "+v"(w[6]), "+v"(w[7]));
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = voxel_value<DT>(w[i]);
    return lerp8(v, f.fx, f.fy, f.fz, true);
  }
  // the same of a channel that differs between lanes
  __device__ __forceinline__ float sample_lane(V3 p, int c) const {
    if (p.x < 0.0f || p.x > 1.0f || p.y < 0.0f || p.y > 1.0f || p.z < 0.0f || p.z > 1.0f)
      return qnan();
    return trilinear(corners(p, c));
  }

  // transferFunction (deviceCode.cu:27-42), opacity only; colour is looked
  // up only for the accepted collision (same lerp, same texels). The two
  // divisions by per-channel constants are products with their reciprocals.
  __device__ __forceinline__ float tf_alpha(float f, int c, float& r2out) const {
    const ChanTf t = chtf[c];
    if (f < t.dlo || f > t.dhi) {
      r2out = qnan();
      return 0.0f;
    }
    const float r1 = (f - t.dlo) * t.idw;
    const float r2 = (r1 - t.xlo) * t.ixw;
    r2out = r2;
    return tf_lerp_alpha(tf + t.off, t.n, r2) * t.os;
  }
  // full transferFunction (deviceCode.cu:27-42) for the blend and marcher
  // modes; f is never NaN here (callers test the unit cube or the sample)
  __device__ __forceinline__ float4 tf_rgba(float f, const ChanTf& t) const {
    if (f < t.dlo || f > t.dhi) return make_float4(1.f, 0.f, 1.f, 0.f);
    const float r1 = (f - t.dlo) * t.idw;
    const float r2 = (r1 - t.xlo) * t.ixw;
    float4 v = tf_lerp(tf + t.off, t.n, r2);
    v.w = v.w * t.os;
    return v;
  }
  // calculateGradient (deviceCode.cu:243-281): central differences of the
  // channel's TF opacity, one-sided at the faces of the unit cube
  __device__ V3 gradient(V3 p, float eps, int c) const {
    const float pc[3] = {p.x, p.y, p.z};
    float g[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      float p1[3] = {pc[0], pc[1], pc[2]}, p2[3] = {pc[0], pc[1], pc[2]};
      p1[i] -= eps;
      p2[i] += eps;
      float div;
      if (p1[i] < 0.0f) {
        p1[i] = pc[i];
        p2[i] = pc[i] + eps;
        div = eps;
      } else if (p2[i] > 1.0f) {
        p1[i] = pc[i] - eps;
        p2[i] = pc[i];
        div = eps;
      } else {
        div = 2.0f * eps;
      }
      float r;
      const float v1 = tf_alpha(sample_lane(v3(p1[0], p1[1], p1[2]), c), c, r);
      const float v2 = tf_alpha(sample_lane(v3(p2[0], p2[1], p2[2]), c), c, r);
      g[i] = (v2 - v1) / div;
    }
    return v3(g[0], g[1], g[2]);
  }
  __device__ __forceinline__ void tf_rgb(float r2, int c, HitRec& h) const {
    const ChanTf t = chtf[c];
    if (r2 != r2) {  // outside the value domain: (1, 0, 1, 0)
      h.r = 1.f;
      h.g = 0.f;
      h.b = 1.f;
      return;
    }
    const float4 v = tf_lerp(tf + t.off, t.n, r2);
    h.r = v.x;
    h.g = v.y;
    h.b = v.z;
  }
};

// Transfer-function texels and per-channel TF parameters -> LDS (the caller
// synchronises the workgroup afterwards).
__device__ __forceinline__ void load_tf_lds(const RenderParams& P, float4* s_tf, ChanTf* s_ch) {
  const int C = P.vol.channels;
  const float4* g = reinterpret_cast<const float4*>(P.tf.tab);
  const int total = C * P.tf.stride;
  for (int i = threadIdx.x; i < total; i += blockDim.x) s_tf[i] = g[i];
  if (int(threadIdx.x) < C) {
    const int c = threadIdx.x;
    ChanTf t;
    t.dlo = P.tf.dom_lo[c];
    t.dhi = P.tf.dom_hi[c];
    t.xlo = P.tf.xf_lo[c];
    t.ixw = 1.0f / (P.tf.xf_hi[c] - P.tf.xf_lo[c]);
    t.os = P.tf.opacity[c];
    t.n = P.tf.n[c];
    t.off = c * P.tf.stride;
    t.idw = 1.0f / (P.tf.dom_hi[c] - P.tf.dom_lo[c]);
    s_ch[c] = t;
  }
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ void flush_counts(const RenderParams& P, const Counts& cnt) {
  const uint32_t s = wave_sum(cnt.samples), v = wave_sum(cnt.visits);
  const uint32_t r = wave_sum(cnt.rejections), n = wave_sum(cnt.rays);
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&P.fr.counters[0], (unsigned long long)s);
    atomicAdd(&P.fr.counters[1], (unsigned long long)v);
    atomicAdd(&P.fr.counters[2], (unsigned long long)r);
    atomicAdd(&P.fr.counters[3], (unsigned long long)n);
  }
}

// Workgroup -> 16x16 pixel block (index into the Hilbert block order).
// Workgroups are dispatched round-robin over the 8 XCDs (workgroup i runs on
// XCD i % 8), so the identity map deals consecutive Hilbert blocks to
// different XCDs: every XCD gets an even share of the heavy image regions
// (giving each XCD a contiguous run instead left half of them idle for half
// the frame: the volume's footprint is not spread evenly along the curve),
// and each XCD still works along the curve, every 8th block. Dealing runs of
// 2, 4, 8 or 16 consecutive blocks to each XCD in turn (more L2 sharing
// between neighbouring blocks) measured 0.5-2% slower on 4 x 256^3 u8 at
// 1024^2.
__device__ __forceinline__ uint32_t block_slot(uint32_t b, uint32_t /*n*/) { return b; }

// running mean of the colour (deviceCode.cu:463-469) and, when m2 is set, of
// its square (an addition for confidence intervals and the error estimate;
// off by default, so a plain frame moves only the accumulator's 32 bytes per
// pixel)
__device__ __forceinline__ void accumulate_pixel(const RenderParams& P, void* accum, void* m2,
                                                 uint32_t accum_id, uint32_t pixel, float fr,
                                                 float fg, float fb, float fa) {
  float4* acc = reinterpret_cast<float4*>(accum) + pixel;
  if (P.fr.accumulate) {
    const float k = float(accum_id);
    const float k1 = float(accum_id + 1);
    const float4 a = *acc;
    *acc = make_float4((fr + k * a.x) / k1, (fg + k * a.y) / k1, (fb + k * a.z) / k1,
                       (fa + k * a.w) / k1);
  } else {
    *acc = make_float4(fr, fg, fb, fa);
  }
  if (m2) {
    float4* sq = reinterpret_cast<float4*>(m2) + pixel;
    const float4 q = make_float4(fr * fr, fg * fg, fb * fb, fa * fa);
    if (P.fr.accumulate) {
      const float k = float(accum_id);
      const float k1 = float(accum_id + 1);
      const float4 m = *sq;
      *sq = make_float4((q.x + k * m.x) / k1, (q.y + k * m.y) / k1, (q.z + k * m.z) / k1,
                        (q.w + k * m.w) / k1);
    } else {
      *sq = q;
    }
  }
}

// Shading of one sample (deviceCode.cu:411-433): diffuse, specular and shadow
// factors from the caller (1, 0, 1 without gradient shading and shadows),
// the hit channel's material specular colour, then over the background.
__device__ __forceinline__ void composite_sample(const RenderParams& P, bool hit, float hr,
                                                 float hg, float hb, float ha, float diffuse,
                                                 float specular, float shadow, int ch, float& fr,
                                                 float& fg, float& fb, float& fa) {
  float cr = 0.f, cg = 0.f, cb = 0.f, ca = 0.f;
  if (hit) {
    const float ld = diffuse * shadow * P.fr.light_intensity;
    const float ls = specular * shadow * P.fr.light_intensity;
    const float* sc = P.fr.sh.spec[ch];
    const float mr = hr * 0.75f + sc[0] * 0.25f;
    const float mg = hg * 0.75f + sc[1] * 0.25f;
    const float mb = hb * 0.75f + sc[2] * 0.25f;
    cr = ld * hr + ls * mr + P.fr.ambient * mr;
    cg = ld * hg + ls * mg + P.fr.ambient * mg;
    cb = ld * hb + ls * mb + P.fr.ambient * mb;
    ca = ha;
  }
  // over(color, (bg, 1)) (deviceCode.cu:54-59, 433)
  fr = fr + (cr + P.fr.bg[0] * 1.f * (1.f - ca));
  fg = fg + (cg + P.fr.bg[1] * 1.f * (1.f - ca));
  fb = fb + (cb + P.fr.bg[2] * 1.f * (1.f - ca));
  fa = fa + (ca + (1.f - ca) * 1.f);
}

// Divides the pixel sums (alpha started at 1) by spp and accumulates.
// What one pixel block needs from its view: camera, size, samples, seed,
// frame / accumulation ids and accumulators.
struct ViewCtx {
  const CameraParams* cam;
  int W, H, spp;
  uint32_t seed, frame_id, accum_id;
  void* accum;
  void* m2;
};

__device__ __forceinline__ void finish_pixel(const RenderParams& P, void* accum, void* m2,
                                             uint32_t accum_id, int spp_i, uint32_t pixel,
                                             float fr, float fg, float fb, float fa) {
  const float spp = float(spp_i);
  accumulate_pixel(P, accum, m2, accum_id, pixel, fr / spp, fg / spp, fb / spp, fa / spp);
}

}  // namespace mdwt
