// Host-side launchers of the denoiser kernels (kernels_denoise.hip), used by
// denoise_api.cpp. Tensors are NHWC: element (pixel p, channel c) of a tensor
// with channel stride s and channel offset o is at p * s + o + c. bf16 values
// are stored as uint16_t.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace mdwt {
namespace dn {

// values per pixel of the network input for a volume of `channels` channels:
// rgb, first-hit depth, transmittance, the hit fraction of each channel, the
// standard error of the pixel mean and log2 of the frame count (both scaled)
constexpr int input_width(int channels) { return 7 + channels; }
// kernel-predicting output: kKernel x kKernel filter weights per pixel
constexpr int kKernelRadius = 3;
constexpr int kKernel = 2 * kKernelRadius + 1;
constexpr int kTaps = kKernel * kKernel;
constexpr int kLogitStride = 64;  // logits per pixel, padded to the conv's N tiles
static_assert(kTaps <= kLogitStride, "logit stride");

// largest number of pixels in one launch (a handle's image, a training batch):
// element offsets then fit in 32 bits
constexpr size_t kMaxPixels = size_t(1) << 24;
constexpr int kLayers = 11;

// 3x3 convolution (zero padding) of nimg images of H x W pixels as an implicit
// GEMM on the matrix cores. w: bf16 [9][cout_pad][cin]; cin % 8 == 0,
// cout_pad % 32 == 0, xs and xo multiples of 8. Writes channels < cout of y16
// (bf16) and/or y32 (fp32).
//
// Input sources and epilogues:
// kSrcPlain reads x; kSrcUpCat reads channel c < cu from xl (H/2 x W/2,
// stride cu) at (y / 2, x / 2) and channel c >= cu from x at c - cu (the
// U-Net's nearest upsample and concatenation); kSrcF32 reads the fp32
// network input kin (inputs values per pixel, zero up to cin) as
// pack_input would convert it. kEpiPlain stores y16 / y32;
// kEpiPool also stores the 2 x 2 mean of y16 into pool16 (stride ps), as
// pool() would; kEpiKpn (cout_pad == kLogitStride) applies the
// kernel-predicting filter to kin and writes pred instead of the logits.
// H and W even for kSrcUpCat and kEpiPool; xs, xo, cu multiples of 8.
constexpr int kSrcPlain = 0, kSrcUpCat = 1, kSrcF32 = 2;
// For training: kEpiKpnLoss (as kEpiKpn, bias allowed) writes the bf16 gradient of
// inv_count[image] * squared error with respect to the logits to y16 (stride
// kLogitStride) and adds the squared error to err; the gradient epilogues
// (no bias; act: bf16 layer output whose ReLU the gradient passes): kEpiMask
// writes y16 = bf16(value where act > 0) (act and y16 of stride ys); kEpiUpGrad
// the same of the 2 x 2 sums of channels < cu (act and y16 of stride cu, half
// resolution) and channels >= cu to y32 (stride ys); kEpiPoolGrad the same of
// skip + value / 4 for the 2 x 2 pixels of twice the resolution (skip, act and
// y16 of stride ys).
constexpr int kEpiPlain = 0, kEpiPool = 1, kEpiKpn = 2, kEpiMask = 3, kEpiUpGrad = 4,
              kEpiPoolGrad = 5, kEpiKpnLoss = 6;
struct ConvArgs {
  const uint16_t* x;
  int xs, xo;
  const uint16_t* xl;
  int cu;
  int nimg, H, W, cin;
  const uint16_t* w;
  const float* bias;
  int cout, cout_pad;
  uint16_t* y16;
  float* y32;
  int ys, yo, relu;
  uint16_t* pool16;
  int ps;
  const float* kin;
  int inputs;
  float* pred;
  const uint16_t* act;
  const float* skip;
  const float* target;     // fp32 [pixels][3]
  const float* inv_count;  // one per image
  float* err;
};
hipError_t conv(const ConvArgs& a, int src, int epi, hipStream_t s);
// dw [9][cout][cin] += sum over pixels of g[p][co] * x[p + tap][ci], and behind
// it [cout] += sum over pixels of g[p][co] (the bias gradient), over nimg images.
// g: bf16, channel stride gs (the masked output gradient); x, xl, cu as in
// ConvArgs (cu 0: x alone, cu % 32 == 0); part: scratch of part_cap floats (at
// least 9 * cout * cin + cout). Strides and xo are multiples of 4 and the rows
// hold cin (cout) rounded up to 4 channels, zero past the last.
struct WgradArgs {
  const uint16_t* g;
  int gs;
  const uint16_t* x;
  int xs, xo;
  const uint16_t* xl;
  int cu;
  int nimg, H, W, cin, cout;
  float* part;
  int xc;  // cin rounded up to 4 (set by wgrad)
};
hipError_t wgrad(WgradArgs a, float* dw, size_t part_cap, hipStream_t s);
hipError_t pool(const uint16_t* x, int H, int W, int C, uint16_t* y, hipStream_t s);
hipError_t up(const uint16_t* x, int H, int W, int C, uint16_t* y, int ys, int yo, hipStream_t s);
hipError_t copy_slice(const uint16_t* x, int xs, int xo, int n, int C, uint16_t* y, int ys, int yo,
                      hipStream_t s);
// in: fp32 [n][inputs] -> x: bf16 [n][in_pad], channels from inputs up zero
hipError_t pack_input(const float* in, int n, int inputs, int in_pad, uint16_t* x, hipStream_t s);
// pred [H*W][3] = softmax(logits) over the kTaps neighbourhood of the input
// colour (in: fp32 [H*W][inputs], rgb first; logits: fp32 [H*W][kLogitStride])
hipError_t kpn_apply(const float* in, int inputs, const float* logits, int H, int W, float* pred,
                     hipStream_t s);
hipError_t adam(float* w, const float* g, float* m, float* v, int n, float lr, float b1, float b2,
                float c1, float c2, float eps, hipStream_t s);
// bf16 layouts of every layer's fp32 weights
struct LayoutArgs {
  struct Layer {
    const float* w;
    uint16_t *wf, *wd;
    int cin, cout, cin_pad, cout_pad, cin_pad32;
  } layer[kLayers];
};
hipError_t weight_layouts(const LayoutArgs& a, hipStream_t s);

}  // namespace dn
}  // namespace mdwt
