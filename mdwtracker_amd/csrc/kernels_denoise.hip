// Kernels of the learned denoiser (a 3-level U-Net of 3x3 convolutions): BF16
// activations and weights, FP32 accumulation on the matrix cores
// (v_mfma_f32_32x32x16_bf16), FP32 gradients and Adam state. No reference
// counterpart (the reference renders plain accumulation only).
//
// Tensors are NHWC with a channel stride (so that a convolution can read or
// write a slice of a concatenated tensor). A 3x3 convolution is an implicit
// GEMM: M = pixels, N = output channels, K = 9 taps x input channels. One
// wave computes 32-pixel x 32-channel tiles; the MFMA lane layouts are
//   A (32 x 8):  lane l holds A[l % 32][(l / 32) * 4 + j], j = 0..3
//   B (8 x 32):  lane l holds B[(l / 32) * 4 + j][l % 32]
//   D (32 x 32): lane l, register v holds D[(v / 4) * 8 + (l / 32) * 4 + v % 4][l % 32]
// (checked on the device with known matrices), and for the 16-deep K step
// lane l holds K entries (l / 32) * 8 + j, j = 0..7, of its A row and B
// column (the sum over K does not depend on which entries a lane holds, as
// long as A and B agree), with the same D layout.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "denoise_internal.hpp"

namespace mdwt {
namespace dn {
namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
// fp32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32: two per instruction)
typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f2bf2(float lo, float hi) {
  const bf2v v = {__bf16(lo), __bf16(hi)};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ uint16_t f2bf(float f) { return uint16_t(f2bf2(f, 0.f)); }

// 4 consecutive bf16 (8 bytes, 8-byte aligned) or zeros
__device__ __forceinline__ uint2 load4(const uint16_t* p, bool ok) {
  return ok ? *reinterpret_cast<const uint2*>(p) : make_uint2(0u, 0u);
}

// Kernel-predicting output (Bako et al. 2017): per pixel, the softmax of
// the kTaps logits (fp32 [n][kLogitStride]) weighs the input colour of the
// kKernel x kKernel neighbourhood (coordinates clamped to the image).
__device__ __forceinline__ int kpn_neighbour(int py, int px, int j, int H, int W) {
  const int sy = min(max(py + j / kKernel - kKernelRadius, 0), H - 1);
  const int sx = min(max(px + j % kKernel - kKernelRadius, 0), W - 1);
  return sy * W + sx;
}
// softmax weights of one pixel's logits z into w (unnormalised) and their sum
__device__ __forceinline__ float kpn_weights_z(const float* z, float* w) {
  float m = z[0];
#pragma unroll
  for (int j = 1; j < kTaps; ++j) m = fmaxf(m, z[j]);
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < kTaps; ++j) {
    w[j] = __expf(z[j] - m);
    sum += w[j];
  }
  return sum;
}
// out[0..2] = sum_j softmax(z)_j * rgb(neighbour j) for pixel (py, px)
__device__ __forceinline__ void kpn_filter(const float* __restrict__ in, int inputs, const float* z,
                                           int py, int px, int H, int W, float* out) {
  float w[kTaps];
  const float inv = 1.f / kpn_weights_z(z, w);
  float r = 0.f, g = 0.f, b = 0.f;
#pragma unroll
  for (int j = 0; j < kTaps; ++j) {
    const float* c = in + size_t(kpn_neighbour(py, px, j, H, W)) * inputs;
    r += w[j] * c[0];
    g += w[j] * c[1];
    b += w[j] * c[2];
  }
  out[0] = r * inv;
  out[1] = g * inv;
  out[2] = b * inv;
}

// y = conv3x3(x) (+ bias, ReLU) on v_mfma_f32_32x32x16_bf16: weights w
// [9][cout_pad][cin] (tap-major, K contiguous); output channel n of pixel p
// to y16[p * ys + yo + n] (bf16) and/or y32[p * ys + yo + n] (fp32, fp32);
// channels n >= cout are not written.
//
// A workgroup (4 waves, WX along x by WR along rows) computes R = 2 WR image
// rows x TP = 32 WX pixels x TN = 32 NT output channels; each wave 2 rows x
// 32 pixels x TN channels (2 NT accumulators of 32 x 32). Per chunk of 32
// input channels the workgroup stages the R + 2 halo rows (TP + 2 pixels) and
// the 9 taps' weights of its TN channels in LDS, one 16-byte granule (8
// channels) per load; the next chunk's granules are loaded into registers
// while the current one is multiplied (one barrier pair per chunk). LDS rows
// hold 32 channels padded to 40 bf16 (80 bytes): 16-byte reads stay aligned
// and any 8 consecutive rows cover the 32 banks once. With 16-channel K
// steps, lane l supplies channels (l / 32) * 8 .. + 7 of its pixel (A) and of
// its output channel's weights (B); D is the 32 x 32 layout above.
//
// Input sources: kSrcPlain reads x (stride xs, offset xo). kSrcUpCat reads
// channel c < cu from xl, the tensor at half resolution (stride cu), at the
// pixel (y / 2, x / 2) (nearest upsampling), and channel c >= cu from x at
// c - cu: the U-Net's upsample-and-concatenate without materialising it.
// Epilogues: kEpiPlain stores as above. kEpiPool also writes the 2 x 2 mean of
// the stored bf16 output to pool16 (stride ps), as pool_kernel computes it.
// kEpiKpn stages the fp32 logits of the tile in LDS and applies the
// kernel-predicting filter (as kpn_apply_kernel) to write pred directly.
// Training (a batch of nimg images, each with its own zero border):
// kEpiKpnLoss goes on from the filtered colour to the squared error against
// target (summed into err) and its gradient with respect to the logits, stored
// as the bf16 the backward convolutions read; the three gradient epilogues turn
// an input gradient straight into the next layer's masked bf16 gradient
// (act > 0 is the ReLU's derivative there): kEpiMask at the same resolution;
// kEpiUpGrad through the upsampling (channels < cu: the 2 x 2 sum) and the skip
// (channels >= cu: fp32 to y32); kEpiPoolGrad through the 2 x 2 mean, onto the
// skip's fp32 gradient. No fp32 gradient of an activation but the two skips'
// goes through memory, and no element-wise kernel is left in the step.
constexpr int kChunk = 32;   // input channels per staged chunk
constexpr int kPitch = 40;   // LDS row (bf16): 32 channels + 8 padding
constexpr int kZPitch = kLogitStride + 1;  // LDS row (fp32) of one pixel's logits
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ bf8 lds_frag(const uint16_t* p) {
  return __builtin_bit_cast(bf8, *reinterpret_cast<const uint4*>(p));
}

template <int WX, int WR, int NT>
struct ConvShape {
  static constexpr int RW = 2, R = RW * WR, TP = 32 * WX, XP = TP + 2, TN = 32 * NT;
  static constexpr int kARows = (R + 2) * XP;             // staged pixels
  static constexpr int kAGr = kARows * 4, kBGr = 9 * TN * 4;  // 16-byte granules
  static constexpr int kAPer = (kAGr + 255) / 256, kBPer = (kBGr + 255) / 256;
  static constexpr int kLds = (kARows + 9 * TN) * kPitch;  // bf16
};

// kpn_filter with the colours read from a staged tile: rgb points at the
// pixel's top-left neighbour in a [rows][pitch][3] block of clamped input
// colours (the same values kpn_neighbour would fetch), same arithmetic
__device__ __forceinline__ void kpn_filter_tile(const float* z, const float* rgb, int pitch,
                                                float* out) {
  float w[kTaps];
  const float inv = 1.f / kpn_weights_z(z, w);
  float r = 0.f, g = 0.f, b = 0.f;
#pragma unroll
  for (int j = 0; j < kTaps; ++j) {
    const float* c = rgb + ((j / kKernel) * pitch + j % kKernel) * 3;
    r += w[j] * c[0];
    g += w[j] * c[1];
    b += w[j] * c[2];
  }
  out[0] = r * inv;
  out[1] = g * inv;
  out[2] = b * inv;
}

// The filtered colour of one pixel as kpn_filter_tile gives it, its squared
// error against target (returned) and the gradient of inv_count times the
// error with respect to the logits, dz_j = w_j (c_j - pred) . gpred with gpred
// = 2 inv_count (pred - target), as bf16 into gz (zero past kTaps). The logits z
// (in LDS) are overwritten by their weights: kept in registers, the 49 weights
// spilled 95 VGPRs.
__device__ __forceinline__ float kpn_loss_tile(float* z, const float* rgb, int pitch,
                                               const float* target, float inv_count, uint16_t* gz) {
  float m = z[0];
  for (int j = 1; j < kTaps; ++j) m = fmaxf(m, z[j]);
  float sum = 0.f, r = 0.f, g = 0.f, b = 0.f;
#pragma unroll 7
  for (int j = 0; j < kTaps; ++j) {
    const float w = __expf(z[j] - m);
    z[j] = w;
    sum += w;
    const float* c = rgb + ((j / kKernel) * pitch + j % kKernel) * 3;
    r += w * c[0];
    g += w * c[1];
    b += w * c[2];
  }
  const float inv = 1.f / sum;
  const float pr = r * inv, pg = g * inv, pb = b * inv;
  const float dr = pr - target[0], dg = pg - target[1], db = pb - target[2];
  const float s = 2.f * inv_count;
  const float gr = s * dr, gg = s * dg, gb = s * db;
  const float base = pr * gr + pg * gg + pb * gb;
#pragma unroll
  for (int j0 = 0; j0 < kLogitStride; j0 += 8) {
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int j = j0 + e;
      v[e] = 0.f;
      if (j < kTaps) {
        const float* c = rgb + ((j / kKernel) * pitch + j % kKernel) * 3;
        v[e] = z[j] * inv * (c[0] * gr + c[1] * gg + c[2] * gb - base);
      }
    }
    *reinterpret_cast<uint4*>(gz + j0) =
        make_uint4(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]), f2bf2(v[4], v[5]), f2bf2(v[6], v[7]));
  }
  return dr * dr + dg * dg + db * db;
}

// lane l ^ 1's value (DPP quad_perm [1, 0, 3, 2])
__device__ __forceinline__ float lane_xor1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false));
}
// 4 gradient values through a ReLU whose output is act, as bf16
__device__ __forceinline__ void store_masked(uint16_t* y, const uint16_t* act, const float v[4]) {
  const uint2 k = *reinterpret_cast<const uint2*>(act);
  const float m0 = bf2f(uint16_t(k.x)) > 0.f ? v[0] : 0.f, m1 = bf2f(uint16_t(k.x >> 16)) > 0.f ? v[1] : 0.f;
  const float m2 = bf2f(uint16_t(k.y)) > 0.f ? v[2] : 0.f, m3 = bf2f(uint16_t(k.y >> 16)) > 0.f ? v[3] : 0.f;
  *reinterpret_cast<uint2*>(y) = make_uint2(f2bf2(m0, m1), f2bf2(m2, m3));
}

// The MFMAs of one staged chunk for waves of one 32-channel tile: 9 taps x
// STEPS K16 steps, fully unrolled, with the next step's LDS fragments read
// before the current step's MFMAs are issued (two fragment sets in
// registers). Waves of two or three tiles have no registers to spare for
// the second set and run the tap loop in the kernel.
template <int WX, int WR, int NT, int STEPS>
__device__ __forceinline__ void mma_chunk(const uint16_t* sA, const uint16_t* sB, int wr, int wx,
                                          int r32, int kh, f16v (&acc)[2][NT]) {
  using S = ConvShape<WX, WR, NT>;
  constexpr int RW = S::RW, XP = S::XP, TN = S::TN, NS = 9 * STEPS;
  const uint16_t* ab = &sA[((wr * RW) * XP + wx * 32 + r32) * kPitch + kh];
  const uint16_t* bb = &sB[r32 * kPitch + kh];
  bf8 fa[2][RW], fb[2][NT];
  auto load = [&](int i, int buf) {
    const int tap = i / STEPS, st = i % STEPS, dyi = tap / 3, dx = tap % 3;
#pragma unroll
    for (int j = 0; j < NT; ++j) fb[buf][j] = lds_frag(bb + (tap * TN + j * 32) * kPitch + 16 * st);
#pragma unroll
    for (int r = 0; r < RW; ++r) fa[buf][r] = lds_frag(ab + ((r + dyi) * XP + dx) * kPitch + 16 * st);
  };
  load(0, 0);
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    if (i + 1 < NS) load(i + 1, (i + 1) & 1);
#pragma unroll
    for (int r = 0; r < RW; ++r)
      acc[r][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[i & 1][0], fa[i & 1][r], acc[r][0], 0, 0, 0);
    // keep the schedule to one step ahead (hoisting every read would need
    // all fragments in registers at once)
    __builtin_amdgcn_sched_barrier(0);
  }
}

// bias of channels n .. n + 3 (0 past cout or without bias); n % 4 == 0
__device__ __forceinline__ float4 bias4(const float* bias, int n, int cout) {
  if (!bias || n >= cout) return make_float4(0.f, 0.f, 0.f, 0.f);
  if (n + 3 < cout) return *reinterpret_cast<const float4*>(bias + n);
  return make_float4(bias[n], n + 1 < cout ? bias[n + 1] : 0.f, n + 2 < cout ? bias[n + 2] : 0.f, 0.f);
}

template <int WX, int WR, int NT, int SRC, int EPI>
__global__ __launch_bounds__(256, 2) void conv_kernel(ConvArgs a) {
  using S = ConvShape<WX, WR, NT>;
  constexpr int RW = S::RW, R = S::R, TP = S::TP, XP = S::XP, TN = S::TN;
  constexpr bool kKpn = EPI == kEpiKpn || EPI == kEpiKpnLoss;
  static_assert(!kKpn || (R * TP * kZPitch + (R + 2 * kKernelRadius) *
                                                      (TP + 2 * kKernelRadius) * 3) * 4 <= S::kLds * 2,
                "filter tile");
  __shared__ __align__(16) uint16_t lds[S::kLds];
  uint16_t* sA = lds;
  uint16_t* sB = lds + S::kARows * kPitch;
  const int t = threadIdx.x, l = t & 63, wv = t >> 6;
  const int tiles_x = (a.W + TP - 1) / TP, tiles_img = tiles_x * ((a.H + R - 1) / R);
  const int ntiles = tiles_img * a.nimg;
  const uint32_t img_px = uint32_t(a.H) * uint32_t(a.W);
  const int n0 = blockIdx.y * TN;
  const int wx = wv % WX, wr = wv / WX;
  const int r32 = l & 31, kh = (l >> 5) * 8, kq = (l >> 5) * 4;
  const uint4 zero = {0u, 0u, 0u, 0u};
  // Tiles of this workgroup: with a grid that is a multiple of the 8 XCDs
  // (workgroup i runs on XCD i % 8), XCD x takes the x-th eighth of the
  // tiles (row bands that share halo rows stay in one L2) and its workgroups
  // stride through it; otherwise a plain grid stride.
  int first, stride, last;
  if (gridDim.x % 8 == 0) {
    const int per = int(gridDim.x) / 8, span = (ntiles + 7) / 8, xcd = int(blockIdx.x) % 8;
    first = xcd * span + int(blockIdx.x) / 8;
    stride = per;
    last = min(ntiles, (xcd + 1) * span);
  } else {
    first = blockIdx.x;
    stride = gridDim.x;
    last = ntiles;
  }
  if (first >= last) return;
  // one chunk of input channels: the weights stay in LDS for every tile
  // (not with the filter epilogue, whose logits overwrite them)
  const bool b_once = !kKpn && a.cin <= kChunk;

  uint4 pa[S::kAPer], pb[S::kBPer];
  // kSrcF32: the fp32 network input, 8 values per granule, converted to
  // bf16 when stored to LDS (as pack_input_kernel converts them)
  constexpr int kF32 = SRC == kSrcF32 ? S::kAPer : 1;
  float pf[kF32][8];
  auto fetch = [&](int tile, int kc, bool with_b) {
    const int img = tile / tiles_img, it = tile - img * tiles_img;
    const int y0 = (it / tiles_x) * R, x0 = (it % tiles_x) * TP;
    const uint32_t p0 = uint32_t(img) * img_px;  // first pixel of the image
#pragma unroll
    for (int i = 0; i < S::kAPer; ++i) {
      const int f = t + 256 * i;
      pa[i] = zero;
      if constexpr (SRC == kSrcF32)
#pragma unroll
        for (int e = 0; e < 8; ++e) pf[i][e] = 0.f;
      if (f < S::kAGr) {
        const int g = f & 3, pp = f >> 2, row = pp / XP, px = pp - row * XP;
        const int sy = y0 + row - 1, sx = x0 + px - 1, c = kc + 8 * g;
        if (sy >= 0 && sy < a.H && sx >= 0 && sx < a.W && c < a.cin) {
          if constexpr (SRC == kSrcF32) {
            const float* q =
                a.kin + (p0 + uint32_t(sy) * uint32_t(a.W) + uint32_t(sx)) * uint32_t(a.inputs);
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (c + e < a.inputs) pf[i][e] = q[c + e];
            continue;
          }
          const uint16_t* p;
          if (SRC == kSrcUpCat && c < a.cu)
            p = a.xl + (p0 / 4u + uint32_t(sy >> 1) * uint32_t(a.W >> 1) + uint32_t(sx >> 1)) * uint32_t(a.cu) +
                uint32_t(c);
          else
            p = a.x + (p0 + uint32_t(sy) * uint32_t(a.W) + uint32_t(sx)) * uint32_t(a.xs) +
                uint32_t(a.xo + (SRC == kSrcUpCat ? c - a.cu : c));
          pa[i] = *reinterpret_cast<const uint4*>(p);
        }
      }
    }
    if (!with_b) return;
#pragma unroll
    for (int i = 0; i < S::kBPer; ++i) {
      const int f = t + 256 * i;
      pb[i] = zero;
      if (f < S::kBGr) {
        const int g = f & 3, q = f >> 2, tap = q / TN, n = q - tap * TN, c = kc + 8 * g;
        if (c < a.cin)
          pb[i] = *reinterpret_cast<const uint4*>(
              a.w + (uint32_t(tap) * uint32_t(a.cout_pad) + uint32_t(n0 + n)) * uint32_t(a.cin) + uint32_t(c));
      }
    }
  };
  auto store = [&](bool with_b) {
#pragma unroll
    for (int i = 0; i < S::kAPer; ++i) {
      const int f = t + 256 * i;
      if constexpr (SRC == kSrcF32) {
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          w[e] = f2bf2(pf[i][2 * e], pf[i][2 * e + 1]);
        pa[i] = make_uint4(w[0], w[1], w[2], w[3]);
      }
      if (f < S::kAGr) *reinterpret_cast<uint4*>(&sA[(f >> 2) * kPitch + 8 * (f & 3)]) = pa[i];
    }
    if (!with_b) return;
#pragma unroll
    for (int i = 0; i < S::kBPer; ++i) {
      const int f = t + 256 * i;
      if (f < S::kBGr) *reinterpret_cast<uint4*>(&sB[(f >> 2) * kPitch + 8 * (f & 3)]) = pb[i];
    }
  };

  f16v acc[RW][NT];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[r][j] = f16v{};
  [[maybe_unused]] float err = 0.f;  // kEpiKpnLoss: this thread's squared error
  // stages (tile, chunk) in order; the next stage's granules are loaded while
  // the current one is multiplied and while the finished tile is stored
  int tile = first, kc = 0;
  bool first_stage = true;
  fetch(tile, 0, true);
  while (true) {
    store(first_stage || !b_once);
    first_stage = false;
    __syncthreads();
    int ntile = tile, nkc = kc + kChunk;
    if (nkc >= a.cin) {
      nkc = 0;
      ntile += stride;
    }
    const bool more = ntile < last;
    if (more) fetch(ntile, nkc, !b_once);
    // K16 steps of the chunk (granules past cin are zero): 9 taps x 1 or 2
    if constexpr (NT == 1) {
      if (a.cin - kc > 16)
        mma_chunk<WX, WR, NT, 2>(sA, sB, wr, wx, r32, kh, acc);
      else
        mma_chunk<WX, WR, NT, 1>(sA, sB, wr, wx, r32, kh, acc);
    } else {
      const int steps = a.cin - kc > 16 ? 2 : 1;
#pragma unroll 1
      for (int tap = 0; tap < 9; ++tap) {
        const int dyi = tap / 3, dx = tap - dyi * 3;
        const uint16_t* ar = &sA[((wr * RW + dyi) * XP + wx * 32 + r32 + dx) * kPitch + kh];
        const uint16_t* br = &sB[(tap * TN + r32) * kPitch + kh];
        for (int st = 0; st < steps; ++st) {
          bf8 b[NT];
#pragma unroll
          for (int j = 0; j < NT; ++j) b[j] = lds_frag(br + j * 32 * kPitch + 16 * st);
#pragma unroll
          for (int r = 0; r < RW; ++r) {
            const bf8 av = lds_frag(ar + r * XP * kPitch + 16 * st);
#pragma unroll
            for (int j = 0; j < NT; ++j)
              acc[r][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], av, acc[r][j], 0, 0, 0);
          }
        }
      }
    }
    __syncthreads();
    if (nkc == 0) {  // the tile is complete
      const int img = tile / tiles_img, it = tile - img * tiles_img;
      const int y0 = (it / tiles_x) * R, x0 = (it % tiles_x) * TP;
      const uint32_t p0 = uint32_t(img) * img_px;
      // acc[r][j]: D = weights x pixels, so lane l holds pixel r32 of row
      // y0 + wr * RW + r and, in register v, output channel
      // j * 32 + (v / 4) * 8 + kq + v % 4: four consecutive channels per
      // register group
      const int px = x0 + wx * 32 + r32;
      if constexpr (kKpn) {
        // logits (fp32, kLogitStride per pixel; n0 == 0, TN == kLogitStride)
        // of the tile into LDS, and after them the input colours of the tile
        // with a kKernelRadius halo (coordinates clamped to the image); then
        // one thread per pixel applies the filter
        float* sz = reinterpret_cast<float*>(lds);
        float* srgb = sz + R * TP * kZPitch;
        constexpr int kRgbCols = TP + 2 * kKernelRadius, kRgbPx = (R + 2 * kKernelRadius) * kRgbCols;
        constexpr int kRgbPer = (kRgbPx + 255) / 256;
        float cr[kRgbPer][3];
#pragma unroll
        for (int i = 0; i < kRgbPer; ++i) {
          const int q = t + 256 * i;
          if (q < kRgbPx) {
            const int iy = q / kRgbCols, ix = q - iy * kRgbCols;
            const int sy = min(max(y0 - kKernelRadius + iy, 0), a.H - 1);
            const int sx = min(max(x0 - kKernelRadius + ix, 0), a.W - 1);
            const float* c = a.kin + (size_t(p0) + size_t(sy) * a.W + sx) * a.inputs;
            cr[i][0] = c[0];
            cr[i][1] = c[1];
            cr[i][2] = c[2];
          }
        }
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int gq = 0; gq < 4; ++gq) {
            const int n = j * 32 + gq * 8 + kq;
            const float4 b4 = bias4(a.bias, n, a.cout);
            const float bn[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int r = 0; r < RW; ++r) {
              const int pl = (wr * RW + r) * TP + wx * 32 + r32;
#pragma unroll
              for (int e = 0; e < 4; ++e) sz[pl * kZPitch + n + e] = acc[r][j][gq * 4 + e] + bn[e];
            }
          }
#pragma unroll
        for (int i = 0; i < kRgbPer; ++i) {
          const int q = t + 256 * i;
          if (q < kRgbPx) {
            srgb[q * 3 + 0] = cr[i][0];
            srgb[q * 3 + 1] = cr[i][1];
            srgb[q * 3 + 2] = cr[i][2];
          }
        }
        __syncthreads();
        for (int pl = t; pl < R * TP; pl += 256) {
          const int ly = pl / TP, lx = pl % TP, py = y0 + ly, qx = x0 + lx;
          const bool in = py < a.H && qx < a.W;
          const size_t p = size_t(p0) + size_t(py) * a.W + qx;
          const float* rgb = srgb + (ly * kRgbCols + lx) * 3;
          if constexpr (EPI == kEpiKpn) {
            if (in) kpn_filter_tile(sz + pl * kZPitch, rgb, kRgbCols, a.pred + p * 3);
          } else {
            if (in)
              err += kpn_loss_tile(sz + pl * kZPitch, rgb, kRgbCols, a.target + p * 3,
                                   a.inv_count[img], a.y16 + p * kLogitStride);
          }
        }
        __syncthreads();  // before the next stage overwrites the logits
      } else if constexpr (EPI == kEpiMask || EPI == kEpiUpGrad || EPI == kEpiPoolGrad) {
        const int y = y0 + wr * RW;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int gq = 0; gq < 4; ++gq) {
            const int n = n0 + j * 32 + gq * 8 + kq;  // channels n .. n + 3 (cout % 4 == 0)
            if constexpr (EPI == kEpiMask) {
#pragma unroll
              for (int r = 0; r < RW; ++r) {
                if (y + r >= a.H || px >= a.W || n >= a.cout) continue;
                const uint32_t o = (p0 + uint32_t(y + r) * uint32_t(a.W) + uint32_t(px)) *
                                       uint32_t(a.ys) + uint32_t(n);
                const float v[4] = {acc[r][j][gq * 4], acc[r][j][gq * 4 + 1], acc[r][j][gq * 4 + 2],
                                    acc[r][j][gq * 4 + 3]};
                store_masked(a.y16 + o, a.act + o, v);
              }
            } else if constexpr (EPI == kEpiUpGrad) {
              if (n0 + j * 32 < a.cu) {  // whole 32-channel tiles on either side
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const float u0 = acc[0][j][gq * 4 + e], u1 = acc[1][j][gq * 4 + e];
                  v[e] = u0 + lane_xor1(u0) + u1 + lane_xor1(u1);
                }
                if ((r32 & 1) == 0 && y < a.H && px < a.W) {
                  const uint32_t o = (p0 / 4u + uint32_t(y >> 1) * uint32_t(a.W >> 1) + uint32_t(px >> 1)) *
                                         uint32_t(a.cu) + uint32_t(n);
                  store_masked(a.y16 + o, a.act + o, v);
                }
              } else {
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                  if (y + r >= a.H || px >= a.W || n >= a.cout) continue;
                  const uint32_t o = (p0 + uint32_t(y + r) * uint32_t(a.W) + uint32_t(px)) *
                                         uint32_t(a.ys) + uint32_t(n - a.cu);
                  *reinterpret_cast<float4*>(a.y32 + o) =
                      make_float4(acc[r][j][gq * 4], acc[r][j][gq * 4 + 1], acc[r][j][gq * 4 + 2],
                                  acc[r][j][gq * 4 + 3]);
                }
              }
            } else {
#pragma unroll
              for (int r = 0; r < RW; ++r) {
                if (y + r >= a.H || px >= a.W || n >= a.cout) continue;
                const float v[4] = {acc[r][j][gq * 4], acc[r][j][gq * 4 + 1], acc[r][j][gq * 4 + 2],
                                    acc[r][j][gq * 4 + 3]};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                  const uint32_t o = (4u * p0 + uint32_t(2 * (y + r) + (q >> 1)) * uint32_t(2 * a.W) +
                                      uint32_t(2 * px + (q & 1))) * uint32_t(a.ys) + uint32_t(n);
                  const float4 sk = *reinterpret_cast<const float4*>(a.skip + o);
                  const float u[4] = {sk.x + 0.25f * v[0], sk.y + 0.25f * v[1], sk.z + 0.25f * v[2],
                                      sk.w + 0.25f * v[3]};
                  store_masked(a.y16 + o, a.act + o, u);
                }
              }
            }
          }
      } else {
        const int y = y0 + wr * RW;  // even: R and RW are
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int gq = 0; gq < 4; ++gq) {
            const int n = n0 + j * 32 + gq * 8 + kq;  // channels n .. n + 3
            const float4 b4 = bias4(a.bias, n, a.cout);
            const float bn[4] = {b4.x, b4.y, b4.z, b4.w};
            uint32_t o16[RW][2];  // bf16 pairs (n, n + 1), (n + 2, n + 3)
#pragma unroll
            for (int r = 0; r < RW; ++r) {
              float o32[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                o32[e] = acc[r][j][gq * 4 + e] + bn[e];
                if (a.relu) o32[e] = fmaxf(o32[e], 0.f);
              }
              o16[r][0] = f2bf2(o32[0], o32[1]);
              o16[r][1] = f2bf2(o32[2], o32[3]);
              if (y + r >= a.H || px >= a.W || n >= a.cout) continue;
              // element offsets stay below 2^31 (at most 2^24 pixels x 96
              // channels at full resolution, 160 at half)
              const uint32_t o = (p0 + uint32_t(y + r) * uint32_t(a.W) + uint32_t(px)) * uint32_t(a.ys) +
                                 uint32_t(a.yo + n);
              if (n + 3 < a.cout) {  // 8-byte bf16 / 16-byte fp32 stores
                if (a.y16) *reinterpret_cast<uint2*>(a.y16 + o) = make_uint2(o16[r][0], o16[r][1]);
                if (a.y32)
                  *reinterpret_cast<float4*>(a.y32 + o) = make_float4(o32[0], o32[1], o32[2], o32[3]);
              } else {
                for (int e = 0; n + e < a.cout; ++e) {
                  if (a.y16) a.y16[o + e] = uint16_t(o16[r][e >> 1] >> ((e & 1) * 16));
                  if (a.y32) a.y32[o + e] = o32[e];
                }
              }
            }
            if constexpr (EPI == kEpiPool) {
              // pixel px + 1 is lane l + 1's; even lanes (px even) write the
              // mean of rows y, y + 1 and pixels px, px + 1
              uint32_t nb16[RW][2];
#pragma unroll
              for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int d = 0; d < 2; ++d)  // DPP quad_perm [1, 0, 3, 2]: lane l ^ 1
                  nb16[r][d] = uint32_t(__builtin_amdgcn_mov_dpp(int(o16[r][d]), 0xB1, 0xF, 0xF, false));
              if ((r32 & 1) == 0 && y < a.H && px < a.W && n < a.cout) {
                float mf[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const int d = e >> 1, sh = (e & 1) * 16;
                  const float s = bf2f(uint16_t(o16[0][d] >> sh)) + bf2f(uint16_t(nb16[0][d] >> sh)) +
                                  bf2f(uint16_t(o16[1][d] >> sh)) + bf2f(uint16_t(nb16[1][d] >> sh));
                  mf[e] = 0.25f * s;
                }
                const uint32_t m01 = f2bf2(mf[0], mf[1]), m23 = f2bf2(mf[2], mf[3]);
                const uint32_t o = (p0 / 4u + uint32_t(y >> 1) * uint32_t(a.W >> 1) + uint32_t(px >> 1)) *
                                       uint32_t(a.ps) + uint32_t(n);
                if (n + 3 < a.cout)
                  *reinterpret_cast<uint2*>(a.pool16 + o) = make_uint2(m01, m23);
                else
                  for (int e = 0; n + e < a.cout; ++e)
                    a.pool16[o + e] = uint16_t((e < 2 ? m01 : m23) >> ((e & 1) * 16));
              }
            }
          }
      }
#pragma unroll
      for (int r = 0; r < RW; ++r)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[r][j] = f16v{};
    }
    if (!more) break;
    tile = ntile;
    kc = nkc;
  }
  if constexpr (EPI == kEpiKpnLoss) {
    for (int o = 32; o > 0; o >>= 1) err += __shfl_down(err, o, 64);
    if (l == 0) atomicAdd(a.err, err);
  }
}

// Weight gradient, GEMM M = output channels, N = input channels, K = pixels:
//   part[wg][tap][co][ci] = sum over the workgroup's pixels p of g[p][co] * x[p + tap][ci]
//   part[wg][9 * cout * cin + co] = sum of g[p][co] (the bias gradient)
// g: bf16 [image][H*W][gs] (the masked output gradient), x: the layer's input
// (for a concatenated input the channels < cu are the half-resolution tensor
// xl's, nearest upsampled, so nothing is materialised).
//
// A wave owns one (32 output x 32 input channels) tile with all nine taps
// (9 accumulators of 32 x 32) and walks down units of 32 columns x kUnitRows
// rows of an image: per row it stages one gradient row and one new input row
// (the last two stay in a ring of three), transposed to [channel][pixel], and
// multiplies 2 K steps x 9 taps. The MFMA needs 8 consecutive pixels of a
// channel per lane: a lane loads 4 pixels x 4 channels, transposes them in
// registers (v_perm) and writes 4 pixels of a channel with one 8-byte store;
// the taps' one- and two-pixel shifts are funnel shifts of one 16 + 4-byte read.
// Per row 18 MFMAs stand against about 130 VALU and 30 LDS instructions. The
// next row is loaded into registers while the current one is multiplied; waves
// share nothing until their four sums are added (in order) at the end, so the
// result does not depend on scheduling. The eleven layers of a step on 8 x
// 256^2: 2591 us with one tap row per wave, element-by-element transposed
// staging and an image at a time, 451 us so (124 GFLOP: 275 TFLOP/s), the bias
// sums (753 + 440 us as kernels of their own) included.
// orders a wave's own LDS writes and reads (its lanes exchange rows through it)
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
constexpr int kSeg = 32;       // columns of a unit: 2 MFMA K steps
constexpr int kUnitRows = 8;   // rows of a unit (2 more input rows are staged)
constexpr int kWPitch = 40;    // LDS row: 34 pixels, 16-byte reads, conflict-free as kPitch

// rows (pixels) of 4 channels -> rows (channels) of 4 pixels
__device__ __forceinline__ void transpose4(const uint2 p[4], uint2 c[4]) {
  c[0] = make_uint2(__builtin_amdgcn_perm(p[1].x, p[0].x, 0x05040100u),
                    __builtin_amdgcn_perm(p[3].x, p[2].x, 0x05040100u));
  c[1] = make_uint2(__builtin_amdgcn_perm(p[1].x, p[0].x, 0x07060302u),
                    __builtin_amdgcn_perm(p[3].x, p[2].x, 0x07060302u));
  c[2] = make_uint2(__builtin_amdgcn_perm(p[1].y, p[0].y, 0x05040100u),
                    __builtin_amdgcn_perm(p[3].y, p[2].y, 0x05040100u));
  c[3] = make_uint2(__builtin_amdgcn_perm(p[1].y, p[0].y, 0x07060302u),
                    __builtin_amdgcn_perm(p[3].y, p[2].y, 0x07060302u));
}

__global__ __launch_bounds__(256, 2) void wgrad_kernel(WgradArgs a) {
  constexpr int kRowsG = 32 * kWPitch;  // one staged row of 32 channels
  constexpr int kWave = 4 * kRowsG;     // gradient row + ring of three input rows
  __shared__ __align__(16) uint16_t lds[4 * kWave];
  static_assert(9 * 32 * 32 * 4 + 32 * 4 <= int(sizeof(lds)), "the waves' sums are added in the same LDS");
  const int l = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ci0 = blockIdx.x * 32, co0 = blockIdx.y * 32;
  const int r32 = l & 31, kh = (l >> 5) * 8, kq = (l >> 5) * 4;
  const int pg = l & 7, cg = l >> 3;  // this lane's 4 pixels and 4 channels of a staged row
  uint16_t* sg = lds + wave * kWave;
  uint16_t* sx = sg + kRowsG;
  const bool up = ci0 < a.cu;
  const uint16_t* xb = up ? a.xl + ci0 : a.x + a.xo + ci0 - a.cu;
  const int xs = up ? a.cu : a.xs, sh = up ? 1 : 0, xw = a.W >> sh;
  const bool g_ok = co0 + 4 * cg < a.gs, x_ok = ci0 + 4 * cg < a.xc;
  const int segs = (a.W + kSeg - 1) / kSeg, nb = (a.H + kUnitRows - 1) / kUnitRows;
  const int units = a.nimg * nb * segs;

  f16v acc[9], accb = f16v{};
#pragma unroll
  for (int t = 0; t < 9; ++t) acc[t] = f16v{};
  const bf8 ones = {__bf16(1.f), __bf16(1.f), __bf16(1.f), __bf16(1.f),
                    __bf16(1.f), __bf16(1.f), __bf16(1.f), __bf16(1.f)};

  for (int unit = int(blockIdx.z) * 4 + wave; unit < units; unit += int(gridDim.z) * 4) {
    const int seg = unit % segs, rest = unit / segs, band = rest % nb, img = rest / nb;
    const int x0 = seg * kSeg, y0 = band * kUnitRows, y1 = min(a.H, y0 + kUnitRows);
    const uint16_t* gi = a.g + size_t(img) * a.H * a.W * a.gs + co0 + 4 * cg;
    const uint16_t* xi = xb + size_t(img) * ((a.H >> sh) * size_t(xw)) * xs + 4 * cg;
    uint2 rg[4], rx[4], rh[2];
    auto load_g = [&](int y) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int px = x0 + 4 * pg + i;
        rg[i] = load4(gi + (size_t(y) * a.W + px) * a.gs, g_ok && y < y1 && px < a.W);
      }
    };
    // staged position s of an input row is column x0 - 1 + s, s = 0 .. 33
    auto load_x = [&](int y) {
      const bool row = x_ok && y >= 0 && y < a.H;
      const uint16_t* q = xi + size_t(row ? y >> sh : 0) * xw * xs;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int px = x0 - 1 + 4 * pg + i;
        rx[i] = load4(q + size_t(px >> sh) * xs, row && px >= 0 && px < a.W);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int px = x0 + kSeg - 1 + i;
        rh[i] = load4(q + size_t(px >> sh) * xs, row && pg == 0 && px < a.W);
      }
    };
    auto store_g = [&]() {
      uint2 c[4];
      transpose4(rg, c);
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<uint2*>(sg + (4 * cg + j) * kWPitch + 4 * pg) = c[j];
    };
    auto store_x = [&](int slot) {
      uint16_t* q = sx + slot * kRowsG + 4 * cg * kWPitch;
      uint2 c[4];
      transpose4(rx, c);
#pragma unroll
      for (int j = 0; j < 4; ++j) *reinterpret_cast<uint2*>(q + j * kWPitch + 4 * pg) = c[j];
      if (pg == 0) {
        const uint2 h[4] = {rh[0], rh[1], make_uint2(0u, 0u), make_uint2(0u, 0u)};
        transpose4(h, c);
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<uint32_t*>(q + j * kWPitch + kSeg) = c[j].x;
      }
    };
    int slot = 0;  // ring slot of row y - 1 (y: the row being multiplied)
    load_x(y0 - 1);
    store_x(0);
    load_x(y0);
    store_x(1);
    load_x(y0 + 1);
    load_g(y0);
    for (int y = y0; y < y1; ++y) {
      store_x(slot == 0 ? 2 : slot - 1);  // row y + 1
      store_g();
      wave_lds_sync();
      load_x(y + 2);
      load_g(y + 1);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf8 fg = lds_frag(sg + r32 * kWPitch + 16 * ks + kh);
        if (ci0 == 0) accb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg, ones, accb, 0, 0, 0);
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
          const int sl = slot + dy >= 3 ? slot + dy - 3 : slot + dy;
          const uint16_t* q = sx + sl * kRowsG + r32 * kWPitch + 16 * ks + kh;
          const uint4 w = *reinterpret_cast<const uint4*>(q);
          const uint32_t w4 = *reinterpret_cast<const uint32_t*>(q + 8);
          const uint4 s1 = make_uint4(__builtin_amdgcn_alignbit(w.y, w.x, 16), __builtin_amdgcn_alignbit(w.z, w.y, 16),
                                      __builtin_amdgcn_alignbit(w.w, w.z, 16), __builtin_amdgcn_alignbit(w4, w.w, 16));
          const uint4 s2 = make_uint4(w.y, w.z, w.w, w4);
          acc[dy * 3] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg, __builtin_bit_cast(bf8, w), acc[dy * 3], 0, 0, 0);
          acc[dy * 3 + 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg, __builtin_bit_cast(bf8, s1), acc[dy * 3 + 1], 0, 0, 0);
          acc[dy * 3 + 2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fg, __builtin_bit_cast(bf8, s2), acc[dy * 3 + 2], 0, 0, 0);
        }
      }
      wave_lds_sync();
      slot = slot == 2 ? 0 : slot + 1;
    }
  }
  // the four waves' sums, in order
  float* red = reinterpret_cast<float*>(lds);
  float* redb = red + 9 * 32 * 32;
  for (int w = 0; w < 4; ++w) {
    __syncthreads();
    if (wave == w) {
#pragma unroll
      for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          float* o = red + (t * 32 + (v >> 2) * 8 + kq + (v & 3)) * 32 + r32;
          *o = w == 0 ? acc[t][v] : *o + acc[t][v];
        }
      if (r32 == 0)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          float* o = redb + (v >> 2) * 8 + kq + (v & 3);
          *o = w == 0 ? accb[v] : *o + accb[v];
        }
    }
  }
  __syncthreads();
  float* part = a.part + size_t(blockIdx.z) * (size_t(9) * a.cout * a.cin + a.cout);
  for (int i = threadIdx.x; i < 9 * 32 * 32; i += 256) {
    const int ci = ci0 + (i & 31), co = co0 + ((i >> 5) & 31), t = i >> 10;
    if (ci < a.cin && co < a.cout) part[(size_t(t) * a.cout + co) * a.cin + ci] = red[i];
  }
  if (ci0 == 0 && threadIdx.x < 32 && co0 + int(threadIdx.x) < a.cout)
    part[size_t(9) * a.cout * a.cin + co0 + threadIdx.x] = redb[threadIdx.x];
}

// dw[i] += sum over the workgroups of part[wg][i]. Block: 16 consecutive
// outputs x 16 groups (group g sums workgroups g, g + 16, ...); the groups are
// then added in order, so the result does not depend on scheduling.
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const float* __restrict__ part,
                                                           int bands, int n,
                                                           float* __restrict__ dw) {
  __shared__ float sums[16][17];
  const int t = threadIdx.x, o = t & 15, grp = t >> 4;
  const int i = blockIdx.x * 16 + o;
  float sum = 0.f;
  if (i < n)
    for (int b = grp; b < bands; b += 16) sum += part[size_t(b) * n + i];
  sums[grp][o] = sum;
  __syncthreads();
  if (t < 16 && i < n) {
    float acc = 0.f;
    for (int g2 = 0; g2 < 16; ++g2) acc += sums[g2][t];
    dw[i] += acc;
  }
}

// 2x2 average pool: y[(py, px)] = mean of x over the 2x2 block (bf16, C channels)
__global__ void pool_kernel(const uint16_t* x, int H, int W, int C, uint16_t* y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int h = H / 2, w = W / 2;
  if (i >= h * w * C) return;
  const int c = i % C, q = i / C, qy = q / w, qx = q - qy * w;
  const size_t b = (size_t(2 * qy) * W + 2 * qx) * C + c;
  const float s = bf2f(x[b]) + bf2f(x[b + C]) + bf2f(x[b + size_t(W) * C]) + bf2f(x[b + size_t(W) * C + C]);
  y[i] = f2bf(0.25f * s);
}
// nearest upsample into a channel slice: y[(p)][yo + c] = x[p / 2][c]
__global__ void up_kernel(const uint16_t* x, int H, int W, int C, uint16_t* y, int ys, int yo) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= H * W * C) return;
  const int c = i % C, p = i / C, py = p / W, px = p - py * W;
  y[size_t(p) * ys + yo + c] = x[(size_t(py / 2) * (W / 2) + px / 2) * C + c];
}
// copy a channel slice (bf16): y[p][yo + c] = x[p][xo + c]
__global__ void copy_slice_kernel(const uint16_t* x, int xs, int xo, int n, int C, uint16_t* y,
                                  int ys, int yo) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n * C) return;
  const int c = i % C, p = i / C;
  y[size_t(p) * ys + yo + c] = x[size_t(p) * xs + xo + c];
}
// network input: in (fp32 [n][inputs]) -> bf16 [n][in_pad] (channels from
// inputs up zero)
__global__ void pack_input_kernel(const float* in, int n, int inputs, int in_pad, uint16_t* x) {
  // one thread per 8-channel granule (16-byte store); in_pad % 8 == 0
  const int groups = in_pad / 8;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n * groups) return;
  const int p = i / groups, c0 = (i - p * groups) * 8;
  const float* src = in + size_t(p) * inputs;
  uint32_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = c0 + 2 * e;
    const uint32_t lo = c < inputs ? f2bf(src[c]) : 0u, hi = c + 1 < inputs ? f2bf(src[c + 1]) : 0u;
    w[e] = lo | (hi << 16);
  }
  *reinterpret_cast<uint4*>(x + size_t(p) * in_pad + c0) = make_uint4(w[0], w[1], w[2], w[3]);
}
// pred [n][3] = sum_j softmax(z)_j * rgb(neighbour j)
__global__ void kpn_apply_kernel(const float* __restrict__ in, int inputs,
                                 const float* __restrict__ logits, int H, int W,
                                 float* __restrict__ pred) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= H * W) return;
  const int py = p / W, px = p - py * W;
  kpn_filter(in, inputs, logits + size_t(p) * kLogitStride, py, px, H, W, pred + size_t(p) * 3);
}
// Adam step on fp32 masters (Kingma & Ba 2015), every parameter of the network.
__global__ void adam_kernel(float* w, const float* g, float* m, float* v, int n, float lr,
                            float b1, float b2, float c1, float c2, float eps) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
}

// forward weights [9][cout_pad][cin_pad] (bf16) and dgrad weights
// [9][cin_pad32][cout_pad] = w[8 - tap][co][ci] from the fp32 master
// [9][cout][cin]; padding zero. Layer blockIdx.y.
__global__ void weight_layouts_kernel(LayoutArgs a) {
  const LayoutArgs::Layer& y = a.layer[blockIdx.y];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int nf = 9 * y.cout_pad * y.cin_pad, nd = 9 * y.cin_pad32 * y.cout_pad;
  if (i < nf) {
    const int ci = i % y.cin_pad, r = i / y.cin_pad, co = r % y.cout_pad, tap = r / y.cout_pad;
    y.wf[i] = (ci < y.cin && co < y.cout) ? f2bf(y.w[(size_t(tap) * y.cout + co) * y.cin + ci]) : uint16_t(0);
  }
  if (i < nd) {
    const int co = i % y.cout_pad, r = i / y.cout_pad, ci = r % y.cin_pad32, tap = r / y.cin_pad32;
    y.wd[i] = (ci < y.cin && co < y.cout) ? f2bf(y.w[(size_t(8 - tap) * y.cout + co) * y.cin + ci])
                                          : uint16_t(0);
  }
}

inline unsigned nb(size_t n, unsigned t = 256) { return unsigned((n + t - 1) / t); }

// compute units of the current device (cached per device)
int cu_count() {
  static std::atomic<int> counts[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = counts[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    counts[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

}  // namespace

hipError_t conv(const ConvArgs& a, int src, int epi, hipStream_t s) {
  // 16-byte granules of input and weights
  if (a.cin % 8 || a.cout_pad % 32 || a.xs % 8 || a.xo % 8 || a.ys % 4 || a.yo % 4)
    return hipErrorInvalidValue;
  if (src == kSrcPlain && a.xo + a.cin > a.xs) return hipErrorInvalidValue;
  if (src == kSrcUpCat && (a.cu % 8 || a.cu >= a.cin || a.xo + a.cin - a.cu > a.xs || a.H % 2 ||
                           a.W % 2 || !a.xl))
    return hipErrorInvalidValue;
  if (src == kSrcF32 && (!a.kin || a.inputs > a.cin)) return hipErrorInvalidValue;
  if (epi == kEpiPool && (a.H % 2 || a.W % 2 || !a.pool16 || !a.y16)) return hipErrorInvalidValue;
  const bool kpn = epi == kEpiKpn || epi == kEpiKpnLoss;
  if (kpn && (a.cout_pad != kLogitStride || !a.kin)) return hipErrorInvalidValue;
  if (epi == kEpiKpn && !a.pred) return hipErrorInvalidValue;
  if (epi == kEpiKpnLoss && (!a.target || !a.inv_count || !a.y16 || !a.err)) return hipErrorInvalidValue;
  if (epi >= kEpiMask && epi <= kEpiPoolGrad && (a.cout % 4 || !a.act || !a.y16 || a.bias))
    return hipErrorInvalidValue;
  if (epi == kEpiMask && a.cout > a.ys) return hipErrorInvalidValue;
  if (epi == kEpiUpGrad && (a.cu % 32 || a.cu >= a.cout || a.cout - a.cu > a.ys || a.H % 2 || a.W % 2 ||
                            !a.y32))
    return hipErrorInvalidValue;
  if (epi == kEpiPoolGrad && (a.cout > a.ys || !a.skip)) return hipErrorInvalidValue;
  // 32-bit element offsets, of the pooled gradient's full resolution too
  if (a.nimg < 1 || uint64_t(a.nimg) * a.H * a.W * (epi == kEpiPoolGrad ? 4 : 1) > kMaxPixels)
    return hipErrorInvalidValue;
  // workgroup shape: 2 x 2 waves of 32 pixels x 2 rows (64 pixels x 4 rows),
  // each with 64 output channels, 96 (the 96-channel level) or 32
  const int shape = a.cout_pad % 64 == 0 ? 2 : a.cout_pad % 96 == 0 ? 3 : 1;
  const int TP = 64, R = 4, TN = 32 * shape;
  if (kpn && shape != 2) return hipErrorInvalidValue;
  // a resident grid (two workgroups per CU, one for the 96-channel shape)
  // whose workgroups loop over the tiles
  const int tiles = a.nimg * ((a.W + TP - 1) / TP) * ((a.H + R - 1) / R), ny = a.cout_pad / TN;
  const int resident = std::max(1, cu_count() * (shape == 3 ? 1 : 2) / ny);
  const dim3 grid(unsigned(std::min(tiles, resident)), unsigned(ny));
  const int key = shape * 100 + src * 10 + epi;
  switch (key) {
    case 100: hipLaunchKernelGGL((conv_kernel<2, 2, 1, kSrcPlain, kEpiPlain>), grid, dim3(256), 0, s, a); break;
    case 101: hipLaunchKernelGGL((conv_kernel<2, 2, 1, kSrcPlain, kEpiPool>), grid, dim3(256), 0, s, a); break;
    case 110: hipLaunchKernelGGL((conv_kernel<2, 2, 1, kSrcUpCat, kEpiPlain>), grid, dim3(256), 0, s, a); break;
    case 120: hipLaunchKernelGGL((conv_kernel<2, 2, 1, kSrcF32, kEpiPlain>), grid, dim3(256), 0, s, a); break;
    case 200: hipLaunchKernelGGL((conv_kernel<2, 2, 2, kSrcPlain, kEpiPlain>), grid, dim3(256), 0, s, a); break;
    case 201: hipLaunchKernelGGL((conv_kernel<2, 2, 2, kSrcPlain, kEpiPool>), grid, dim3(256), 0, s, a); break;
    case 202: hipLaunchKernelGGL((conv_kernel<2, 2, 2, kSrcPlain, kEpiKpn>), grid, dim3(256), 0, s, a); break;
    case 210: hipLaunchKernelGGL((conv_kernel<2, 2, 2, kSrcUpCat, kEpiPlain>), grid, dim3(256), 0, s, a); break;
    case 300: hipLaunchKernelGGL((conv_kernel<2, 2, 3, kSrcPlain, kEpiPlain>), grid, dim3(256), 0, s, a); break;
    case 103: hipLaunchKernelGGL((conv_kernel<2, 2, 1, kSrcPlain, kEpiMask>), grid, dim3(256), 0, s, a); break;
    case 104: hipLaunchKernelGGL((conv_kernel<2, 2, 1, kSrcPlain, kEpiUpGrad>), grid, dim3(256), 0, s, a); break;
    case 105: hipLaunchKernelGGL((conv_kernel<2, 2, 1, kSrcPlain, kEpiPoolGrad>), grid, dim3(256), 0, s, a); break;
    case 203: hipLaunchKernelGGL((conv_kernel<2, 2, 2, kSrcPlain, kEpiMask>), grid, dim3(256), 0, s, a); break;
    case 205: hipLaunchKernelGGL((conv_kernel<2, 2, 2, kSrcPlain, kEpiPoolGrad>), grid, dim3(256), 0, s, a); break;
    case 206: hipLaunchKernelGGL((conv_kernel<2, 2, 2, kSrcPlain, kEpiKpnLoss>), grid, dim3(256), 0, s, a); break;
    case 303: hipLaunchKernelGGL((conv_kernel<2, 2, 3, kSrcPlain, kEpiMask>), grid, dim3(256), 0, s, a); break;
    case 304: hipLaunchKernelGGL((conv_kernel<2, 2, 3, kSrcPlain, kEpiUpGrad>), grid, dim3(256), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// workgroups of one weight-gradient launch over all its channel tiles: two per
// CU, one resident round (each adds 36 KiB of partial sums to the reduction)
constexpr int kWgradGroups = 512;

hipError_t wgrad(WgradArgs a, float* dw, size_t part_cap, hipStream_t s) {
  // 8-byte channel groups: strides and offsets in whole groups, and the
  // groups that hold the last channels inside the row
  if (a.gs % 4 || a.xs % 4 || a.xo % 4 || (a.cout + 3) / 4 * 4 > a.gs || a.cu % 32 || a.nimg < 1)
    return hipErrorInvalidValue;
  if (a.cu ? (a.cin % 4 || a.xo + a.cin - a.cu > a.xs || !a.xl || a.H % 2 || a.W % 2)
           : a.xo + (a.cin + 3) / 4 * 4 > a.xs)
    return hipErrorInvalidValue;
  a.xc = (a.cin + 3) / 4 * 4;
  const int tx = (a.cin + 31) / 32, ty = (a.cout + 31) / 32;
  const size_t per = size_t(9) * a.cout * a.cin + a.cout;
  if (per > part_cap) return hipErrorInvalidValue;
  const int units = a.nimg * ((a.H + kUnitRows - 1) / kUnitRows) * ((a.W + kSeg - 1) / kSeg);
  const int groups = std::max(1, std::min({(units + 3) / 4, kWgradGroups / (tx * ty), int(part_cap / per)}));
  hipLaunchKernelGGL(wgrad_kernel, dim3(unsigned(tx), unsigned(ty), unsigned(groups)), dim3(256), 0, s, a);
  hipLaunchKernelGGL(wgrad_reduce_kernel, dim3(nb(per, 16)), dim3(256), 0, s, a.part, groups, int(per), dw);
  return hipGetLastError();
}

hipError_t pool(const uint16_t* x, int H, int W, int C, uint16_t* y, hipStream_t s) {
  hipLaunchKernelGGL(pool_kernel, dim3(nb(size_t(H / 2) * (W / 2) * C)), dim3(256), 0, s, x, H, W,
                     C, y);
  return hipGetLastError();
}
hipError_t up(const uint16_t* x, int H, int W, int C, uint16_t* y, int ys, int yo, hipStream_t s) {
  hipLaunchKernelGGL(up_kernel, dim3(nb(size_t(H) * W * C)), dim3(256), 0, s, x, H, W, C, y, ys,
                     yo);
  return hipGetLastError();
}
hipError_t copy_slice(const uint16_t* x, int xs, int xo, int n, int C, uint16_t* y, int ys, int yo,
                      hipStream_t s) {
  hipLaunchKernelGGL(copy_slice_kernel, dim3(nb(size_t(n) * C)), dim3(256), 0, s, x, xs, xo, n, C,
                     y, ys, yo);
  return hipGetLastError();
}
hipError_t pack_input(const float* in, int n, int inputs, int in_pad, uint16_t* x, hipStream_t s) {
  if (in_pad % 8) return hipErrorInvalidValue;
  hipLaunchKernelGGL(pack_input_kernel, dim3(nb(size_t(n) * (in_pad / 8))), dim3(256), 0, s, in, n,
                     inputs, in_pad, x);
  return hipGetLastError();
}
hipError_t kpn_apply(const float* in, int inputs, const float* logits, int H, int W, float* pred,
                     hipStream_t s) {
  hipLaunchKernelGGL(kpn_apply_kernel, dim3(nb(size_t(H) * W)), dim3(256), 0, s, in, inputs,
                     logits, H, W, pred);
  return hipGetLastError();
}
hipError_t adam(float* w, const float* g, float* m, float* v, int n, float lr, float b1, float b2,
                float c1, float c2, float eps, hipStream_t s) {
  hipLaunchKernelGGL(adam_kernel, dim3(nb(size_t(n))), dim3(256), 0, s, w, g, m, v, n, lr, b1, b2,
                     c1, c2, eps);
  return hipGetLastError();
}
hipError_t weight_layouts(const LayoutArgs& a, hipStream_t s) {
  int n = 0;
  for (const auto& y : a.layer)
    n = std::max({n, 9 * y.cout_pad * y.cin_pad, 9 * y.cin_pad32 * y.cout_pad});
  hipLaunchKernelGGL(weight_layouts_kernel, dim3(nb(size_t(n)), kLayers), dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace dn
}  // namespace mdwt
