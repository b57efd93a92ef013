// Learned denoiser beside plain accumulation: a 3-level U-Net (3x3
// convolutions, 32 / 64 / 96 channels, 2x2 average pooling, nearest
// upsampling with skip concatenation, ReLU), BF16 weights and activations,
// FP32 accumulation on the matrix cores, trained in place with Adam on pairs
// of low- and high-sample renders. Its output is kernel-predicting (Bako et
// al. 2017): per pixel, softmax weights of a 7x7 filter applied to the input
// colour. Input per pixel (7 + channels values): rgb, first-hit depth,
// transmittance, the hit fraction of each channel (mdwt_set_aov), the
// standard error of the pixel mean and log2 of the frame count.
// No reference counterpart; C ABI in include/mdwt_denoise.h.
#include "mdwt_denoise.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "denoise_internal.hpp"
#include "host_copy.hpp"

namespace {

struct Conv {
  int cin = 0, cout = 0;          // real channel counts
  int cin_pad = 0, cout_pad = 0;  // forward layout (K multiple of 8, N multiple of 32)
  int cin_pad32 = 0;              // dgrad N (multiple of 32)
  bool relu = true;
  size_t nw = 0;                  // 9 * cout * cin
  size_t off = 0;                 // of its weights in the parameter arrays, the biases behind them
  float *w = nullptr, *b = nullptr;  // in mdwt_denoiser::params
  uint16_t *wf = nullptr, *wd = nullptr;
};

// What a training step on a batch of `images` images keeps on the device.
// Activations are bf16; gm0 / gm1 hold the masked gradients of two consecutive
// layers, skip1 / skip3 the fp32 gradients of the two skip connections.
struct TrainBufs {
  int images = 0;
  std::vector<void*> bufs;
  float *in32 = nullptr, *tgt = nullptr, *inv = nullptr;
  uint16_t *x0, *a0, *a1, *p1, *a2, *a3, *p2, *a4, *a5, *a6, *a7, *a8, *a9, *gm0, *gm1;
  float *skip1, *skip3;
};

int round_up(int v, int m) { return (v + m - 1) / m * m; }

}  // namespace

struct mdwt_denoiser {
  std::string err;
  int device = 0;
  int H = 0, W = 0;
  int channels = 4, inputs = 11, in_pad = 16;  // input values per pixel, padded to 8
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  Conv c[11];
  std::vector<void*> bufs;
  // fp32 parameters, gradients and Adam moments of every layer: its weights,
  // then its biases (the layout of mdwt_dn_get_params)
  size_t n_params = 0;
  float *params = nullptr, *grads = nullptr, *mom = nullptr, *var = nullptr;
  // inference: activations (bf16) and network io (fp32)
  uint16_t *x0, *a0, *a1, *p1, *a2, *a3, *p2, *a4, *a5, *u2, *a6, *a7, *u1, *a8, *a9;
  float *in32, *out32, *pred, *err_sum;
  float* wpart = nullptr;  // partial weight gradients of the workgroups
  TrainBufs train;  // made by the first step, grown by a larger batch
  int step = 0;
  bool fused = true;  // inference: fused upsample/concat, pooling and filter
};

namespace {

// (as the renderer's: an error of the runtime is reported once)
int fail(mdwt_denoiser* d, int code, const std::string& m) {
  if (code == MDWT_ERR_HIP || code == MDWT_ERR_OOM) (void)hipGetLastError();
  d->err = m;
  return code;
}
#define DNCHK(d, expr)                                                                  \
  do {                                                                                  \
    hipError_t e_ = (expr);                                                             \
    if (e_ != hipSuccess)                                                               \
      return fail((d), MDWT_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

template <class T>
int alloc(mdwt_denoiser* d, T** p, size_t n) {
  void* q = nullptr;
  if (hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)) != hipSuccess)
    return fail(d, MDWT_ERR_OOM, "denoiser allocation");
  d->bufs.push_back(q);
  DNCHK(d, hipMemset(q, 0, std::max<size_t>(n, 1) * sizeof(T)));
  *p = static_cast<T*>(q);
  return MDWT_OK;
}

// layer table: (cin, cout, relu); c0 reads the input (cin set per handle),
// c10 writes the kTaps filter logits
using mdwt::dn::kMaxPixels;  // largest image (pixels) a denoiser handle accepts

const int kLayers[11][3] = {{0, 32, 1}, {32, 32, 1}, {32, 64, 1},
                            {64, 64, 1},  {64, 96, 1}, {96, 96, 1}, {160, 64, 1},
                            {64, 64, 1},  {96, 32, 1}, {32, 32, 1}, {32, mdwt::dn::kTaps, 0}};

// width in pixels of the Gaussian filter the untrained network applies
constexpr float kInitSigma = 1.5f;
// floats of partial weight gradients (48 MiB): at least 9 * cout * cin + cout of
// every layer, and room for enough workgroups to fill the GPU
constexpr size_t kWgradPart = size_t(12) << 20;
// pixels of one training batch on the device (968 bytes each: about 1 GB); larger
// batches go in parts, of one image at least
constexpr size_t kTrainPixels = size_t(1) << 20;

int setup(mdwt_denoiser* d, uint32_t seed) {
  std::mt19937 gen(seed);
  for (int i = 0; i < 11; ++i) {
    Conv& L = d->c[i];
    L.cin = i == 0 ? d->inputs : kLayers[i][0];
    L.cout = kLayers[i][1];
    L.relu = kLayers[i][2] != 0;
    L.cin_pad = i == 0 ? d->in_pad : round_up(L.cin, 8);
    L.cout_pad = round_up(L.cout, 32);
    L.cin_pad32 = round_up(L.cin, 32);
    L.nw = size_t(9) * L.cout * L.cin;
    L.off = d->n_params;
    d->n_params += L.nw + size_t(L.cout);
  }
  int rc;
  if ((rc = alloc(d, &d->params, d->n_params)) || (rc = alloc(d, &d->grads, d->n_params)) ||
      (rc = alloc(d, &d->mom, d->n_params)) || (rc = alloc(d, &d->var, d->n_params)))
    return rc;
  for (int i = 0; i < 11; ++i) {
    Conv& L = d->c[i];
    L.w = d->params + L.off;
    L.b = L.w + L.nw;
    if ((rc = alloc(d, &L.wf, size_t(9) * L.cout_pad * L.cin_pad)) ||
        (rc = alloc(d, &L.wd, size_t(9) * L.cin_pad32 * L.cout_pad)))
      return rc;
    // He initialisation for ReLU layers; the output layer starts small
    // with Gaussian log-weights as bias, so that the untrained network
    // filters with a Gaussian of kInitSigma pixels
    const float sd = L.relu ? std::sqrt(2.f / float(9 * L.cin)) : 1e-3f;
    std::normal_distribution<float> nd(0.f, sd);
    std::vector<float> hw(L.nw);
    for (auto& v : hw) v = nd(gen);
    DNCHK(d, hipMemcpy(L.w, hw.data(), L.nw * sizeof(float), hipMemcpyHostToDevice));
    if (!L.relu) {
      std::vector<float> hb(L.cout);
      for (int j = 0; j < L.cout; ++j) {
        const float dy = float(j / mdwt::dn::kKernel - mdwt::dn::kKernelRadius);
        const float dx = float(j % mdwt::dn::kKernel - mdwt::dn::kKernelRadius);
        hb[j] = -(dx * dx + dy * dy) / (2.f * kInitSigma * kInitSigma);
      }
      DNCHK(d, hipMemcpy(L.b, hb.data(), hb.size() * sizeof(float), hipMemcpyHostToDevice));
    }
  }
  const size_t n = size_t(d->H) * d->W, n4 = n / 4, n16 = n / 16;
  if ((rc = alloc(d, &d->x0, n * d->in_pad)) || (rc = alloc(d, &d->a0, n * 32)) ||
      (rc = alloc(d, &d->a1, n * 32)) || (rc = alloc(d, &d->p1, n4 * 32)) ||
      (rc = alloc(d, &d->a2, n4 * 64)) || (rc = alloc(d, &d->a3, n4 * 64)) ||
      (rc = alloc(d, &d->p2, n16 * 64)) || (rc = alloc(d, &d->a4, n16 * 96)) ||
      (rc = alloc(d, &d->a5, n16 * 96)) || (rc = alloc(d, &d->u2, n4 * 160)) ||
      (rc = alloc(d, &d->a6, n4 * 64)) || (rc = alloc(d, &d->a7, n4 * 64)) ||
      (rc = alloc(d, &d->u1, n * 96)) || (rc = alloc(d, &d->a8, n * 32)) ||
      (rc = alloc(d, &d->a9, n * 32)))
    return rc;
  if ((rc = alloc(d, &d->in32, n * d->inputs)) ||
      (rc = alloc(d, &d->out32, n * mdwt::dn::kLogitStride)) || (rc = alloc(d, &d->pred, n * 3)) ||
      (rc = alloc(d, &d->err_sum, 1)))
    return rc;
  return MDWT_OK;
}

void free_train(TrainBufs* t) {
  for (void* p : t->bufs) (void)hipFree(p);
  *t = TrainBufs{};
}

// Device memory for training on up to `images` images at a time. If it is not
// there for more than the present buffers hold, those stay (and the batch goes
// in smaller parts).
int train_bufs(mdwt_denoiser* d, int images) {
  images = int(std::max<size_t>(1, std::min(size_t(images), kTrainPixels / (size_t(d->H) * d->W))));
  if (images <= d->train.images) return MDWT_OK;
  if (!d->wpart) {
    int rc = alloc(d, &d->wpart, kWgradPart);
    if (rc) return rc;
  }
  while (images > d->train.images) {
    TrainBufs t;
    t.images = images;
    bool ok = true;
    auto get = [&](auto** p, size_t n) {
      void* q = nullptr;
      if (ok && hipMalloc(&q, n * sizeof(**p)) == hipSuccess)
        t.bufs.push_back(q);
      else
        ok = false;
      *p = static_cast<std::remove_reference_t<decltype(*p)>>(q);
    };
    const size_t n = size_t(images) * d->H * d->W, n4 = n / 4, n16 = n / 16;
    get(&t.in32, n * d->inputs);
    get(&t.tgt, n * 3);
    get(&t.inv, size_t(images));
    get(&t.x0, n * d->in_pad);
    get(&t.a0, n * 32);
    get(&t.a1, n * 32);
    get(&t.p1, n4 * 32);
    get(&t.a2, n4 * 64);
    get(&t.a3, n4 * 64);
    get(&t.p2, n16 * 64);
    get(&t.a4, n16 * 96);
    get(&t.a5, n16 * 96);
    get(&t.a6, n4 * 64);
    get(&t.a7, n4 * 64);
    get(&t.a8, n * 32);
    get(&t.a9, n * 32);
    get(&t.gm0, n * mdwt::dn::kLogitStride);
    get(&t.gm1, n * mdwt::dn::kLogitStride);
    get(&t.skip1, n * 32);
    get(&t.skip3, n4 * 64);
    if (ok) {
      free_train(&d->train);
      d->train = std::move(t);
      return MDWT_OK;
    }
    (void)hipGetLastError();
    free_train(&t);
    if (d->train.images > 0) return MDWT_OK;
    if (images == 1) return fail(d, MDWT_ERR_OOM, "denoiser training buffers");
    images = (images + 1) / 2;
  }
  return MDWT_OK;
}

int refresh_weights(mdwt_denoiser* d) {
  mdwt::dn::LayoutArgs a;
  for (int i = 0; i < mdwt::dn::kLayers; ++i) {
    const Conv& L = d->c[i];
    a.layer[i] = {L.w, L.wf, L.wd, L.cin, L.cout, L.cin_pad, L.cout_pad, L.cin_pad32};
  }
  DNCHK(d, mdwt::dn::weight_layouts(a, d->stream));
  return MDWT_OK;
}

// conv layer i forward with an input source / epilogue (ConvArgs)
int fwd_fused(mdwt_denoiser* d, int i, mdwt::dn::ConvArgs a, int src, int epi) {
  const Conv& L = d->c[i];
  a.cin = L.cin_pad;
  a.w = L.wf;
  a.bias = L.b;
  a.cout = L.cout;
  a.cout_pad = L.cout_pad;
  a.relu = L.relu ? 1 : 0;
  DNCHK(d, mdwt::dn::conv(a, src, epi, d->stream));
  return MDWT_OK;
}

mdwt::dn::ConvArgs conv_args(const uint16_t* x, int xs, int nimg, int H, int W, uint16_t* y16, int ys) {
  mdwt::dn::ConvArgs a{};
  a.x = x;
  a.xs = xs;
  a.nimg = nimg;
  a.H = H;
  a.W = W;
  a.y16 = y16;
  a.ys = ys;
  return a;
}

// conv layer i forward: x (stride xs, offset xo) -> y16 / y32 (stride ys)
int fwd(mdwt_denoiser* d, int i, const uint16_t* x, int H, int W, int xs, int xo, uint16_t* y16,
        float* y32, int ys) {
  mdwt::dn::ConvArgs a = conv_args(x, xs, 1, H, W, y16, ys);
  a.xo = xo;
  a.y32 = y32;
  return fwd_fused(d, i, a, mdwt::dn::kSrcPlain, mdwt::dn::kEpiPlain);
}

// Inference with a kernel for every step of the network (mdwt_dn_set_fused 0)

int forward(mdwt_denoiser* d) {
  const int H = d->H, W = d->W, n = H * W;
  const int H2 = H / 2, W2 = W / 2, H4 = H / 4, W4 = W / 4;
  hipStream_t s = d->stream;
  int rc;
  DNCHK(d, mdwt::dn::pack_input(d->in32, n, d->inputs, d->in_pad, d->x0, s));
  if ((rc = fwd(d, 0, d->x0, H, W, d->in_pad, 0, d->a0, nullptr, 32))) return rc;
  if ((rc = fwd(d, 1, d->a0, H, W, 32, 0, d->a1, nullptr, 32))) return rc;
  DNCHK(d, mdwt::dn::pool(d->a1, H, W, 32, d->p1, s));
  if ((rc = fwd(d, 2, d->p1, H2, W2, 32, 0, d->a2, nullptr, 64))) return rc;
  if ((rc = fwd(d, 3, d->a2, H2, W2, 64, 0, d->a3, nullptr, 64))) return rc;
  DNCHK(d, mdwt::dn::pool(d->a3, H2, W2, 64, d->p2, s));
  if ((rc = fwd(d, 4, d->p2, H4, W4, 64, 0, d->a4, nullptr, 96))) return rc;
  if ((rc = fwd(d, 5, d->a4, H4, W4, 96, 0, d->a5, nullptr, 96))) return rc;
  DNCHK(d, mdwt::dn::up(d->a5, H2, W2, 96, d->u2, 160, 0, s));
  DNCHK(d, mdwt::dn::copy_slice(d->a3, 64, 0, H2 * W2, 64, d->u2, 160, 96, s));
  if ((rc = fwd(d, 6, d->u2, H2, W2, 160, 0, d->a6, nullptr, 64))) return rc;
  if ((rc = fwd(d, 7, d->a6, H2, W2, 64, 0, d->a7, nullptr, 64))) return rc;
  DNCHK(d, mdwt::dn::up(d->a7, H, W, 64, d->u1, 96, 0, s));
  DNCHK(d, mdwt::dn::copy_slice(d->a1, 32, 0, n, 32, d->u1, 96, 64, s));
  if ((rc = fwd(d, 8, d->u1, H, W, 96, 0, d->a8, nullptr, 32))) return rc;
  if ((rc = fwd(d, 9, d->a8, H, W, 32, 0, d->a9, nullptr, 32))) return rc;
  if ((rc = fwd(d, 10, d->a9, H, W, 32, 0, nullptr, d->out32, mdwt::dn::kLogitStride))) return rc;
  DNCHK(d, mdwt::dn::kpn_apply(d->in32, d->inputs, d->out32, H, W, d->pred, s));
  return MDWT_OK;
}

// Inference forward: the same values as forward() (every fused step
// computes what the kernel it replaces would have stored), without
// materialising the packed input, the pooled, upsampled and concatenated
// tensors or the logits: c0 converts the fp32 input while staging it, c1
// and c3 pool in their epilogue, c6 and c8 read their two inputs directly,
// c10 applies the filter in its epilogue.
int forward_fused(mdwt_denoiser* d) {
  using namespace mdwt::dn;
  const int H = d->H, W = d->W;
  const int H2 = H / 2, W2 = W / 2, H4 = H / 4, W4 = W / 4;
  int rc;
  auto args = [](const uint16_t* x, int xs, int Hh, int Ww, uint16_t* y16, int ys) {
    return conv_args(x, xs, 1, Hh, Ww, y16, ys);
  };
  ConvArgs a = args(nullptr, 0, H, W, d->a0, 32);  // c0 reads the fp32 input
  a.kin = d->in32;
  a.inputs = d->inputs;
  if ((rc = fwd_fused(d, 0, a, kSrcF32, kEpiPlain))) return rc;
  a = args(d->a0, 32, H, W, d->a1, 32);
  a.pool16 = d->p1;
  a.ps = 32;
  if ((rc = fwd_fused(d, 1, a, kSrcPlain, kEpiPool))) return rc;
  if ((rc = fwd_fused(d, 2, args(d->p1, 32, H2, W2, d->a2, 64), kSrcPlain, kEpiPlain))) return rc;
  a = args(d->a2, 64, H2, W2, d->a3, 64);
  a.pool16 = d->p2;
  a.ps = 64;
  if ((rc = fwd_fused(d, 3, a, kSrcPlain, kEpiPool))) return rc;
  if ((rc = fwd_fused(d, 4, args(d->p2, 64, H4, W4, d->a4, 96), kSrcPlain, kEpiPlain))) return rc;
  if ((rc = fwd_fused(d, 5, args(d->a4, 96, H4, W4, d->a5, 96), kSrcPlain, kEpiPlain))) return rc;
  a = args(d->a3, 64, H2, W2, d->a6, 64);  // channels 0..95: up(a5), 96..159: a3
  a.xl = d->a5;
  a.cu = 96;
  if ((rc = fwd_fused(d, 6, a, kSrcUpCat, kEpiPlain))) return rc;
  if ((rc = fwd_fused(d, 7, args(d->a6, 64, H2, W2, d->a7, 64), kSrcPlain, kEpiPlain))) return rc;
  a = args(d->a1, 32, H, W, d->a8, 32);  // channels 0..63: up(a7), 64..95: a1
  a.xl = d->a7;
  a.cu = 64;
  if ((rc = fwd_fused(d, 8, a, kSrcUpCat, kEpiPlain))) return rc;
  if ((rc = fwd_fused(d, 9, args(d->a8, 32, H, W, d->a9, 32), kSrcPlain, kEpiPlain))) return rc;
  a = args(d->a9, 32, H, W, nullptr, kLogitStride);
  a.kin = d->in32;
  a.inputs = d->inputs;
  a.pred = d->pred;
  return fwd_fused(d, 10, a, kSrcPlain, kEpiKpn);
}

// Backward of conv layer i at B images of H x W: its weight and bias gradients
// from gm (the masked bf16 gradient of its output, stride cout_pad) and its
// input (x, or for a concatenated input xl upsampled and x), then, where epi
// >= 0, the input gradient through epilogue epi of `a` (the target fields).
int bwd(mdwt_denoiser* d, int i, int B, int H, int W, const uint16_t* gm, const uint16_t* x, int xs,
        const uint16_t* xl, int cu, mdwt::dn::ConvArgs a, int epi) {
  const Conv& L = d->c[i];
  mdwt::dn::WgradArgs g{};
  g.g = gm;
  g.gs = L.cout_pad;
  g.x = x;
  g.xs = xs;
  g.xl = xl;
  g.cu = cu;
  g.nimg = B;
  g.H = H;
  g.W = W;
  g.cin = L.cin;
  g.cout = L.cout;
  g.part = d->wpart;
  DNCHK(d, mdwt::dn::wgrad(g, d->grads + L.off, kWgradPart, d->stream));
  if (epi < 0) return MDWT_OK;
  a.x = gm;
  a.xs = L.cout_pad;
  a.nimg = B;
  a.H = H;
  a.W = W;
  a.cin = L.cout_pad;
  a.w = L.wd;
  a.cout = L.cin;
  a.cout_pad = L.cin_pad32;
  DNCHK(d, mdwt::dn::conv(a, mdwt::dn::kSrcPlain, epi, d->stream));
  return MDWT_OK;
}

// Loss gradient of the B images in the training buffers, added to grads (and
// the squared error to err_sum): the forward of forward_fused over the batch,
// keeping the activations, then the layers in reverse. Every kernel takes the
// whole batch: image by image, a step of 8 x 256^2 was about 1000 launches of 5
// to 30 us, most of them too small for the chip: 8.0 ms of kernels, 1.4 ms so.
int train_batch(mdwt_denoiser* d, int B) {
  using namespace mdwt::dn;
  TrainBufs& t = d->train;
  const int H = d->H, W = d->W;
  const int H2 = H / 2, W2 = W / 2, H4 = H / 4, W4 = W / 4;
  int rc;
  DNCHK(d, pack_input(t.in32, B * H * W, d->inputs, d->in_pad, t.x0, d->stream));
  if ((rc = fwd_fused(d, 0, conv_args(t.x0, d->in_pad, B, H, W, t.a0, 32), kSrcPlain, kEpiPlain))) return rc;
  ConvArgs a = conv_args(t.a0, 32, B, H, W, t.a1, 32);
  a.pool16 = t.p1;
  a.ps = 32;
  if ((rc = fwd_fused(d, 1, a, kSrcPlain, kEpiPool))) return rc;
  if ((rc = fwd_fused(d, 2, conv_args(t.p1, 32, B, H2, W2, t.a2, 64), kSrcPlain, kEpiPlain))) return rc;
  a = conv_args(t.a2, 64, B, H2, W2, t.a3, 64);
  a.pool16 = t.p2;
  a.ps = 64;
  if ((rc = fwd_fused(d, 3, a, kSrcPlain, kEpiPool))) return rc;
  if ((rc = fwd_fused(d, 4, conv_args(t.p2, 64, B, H4, W4, t.a4, 96), kSrcPlain, kEpiPlain))) return rc;
  if ((rc = fwd_fused(d, 5, conv_args(t.a4, 96, B, H4, W4, t.a5, 96), kSrcPlain, kEpiPlain))) return rc;
  a = conv_args(t.a3, 64, B, H2, W2, t.a6, 64);
  a.xl = t.a5;
  a.cu = 96;
  if ((rc = fwd_fused(d, 6, a, kSrcUpCat, kEpiPlain))) return rc;
  if ((rc = fwd_fused(d, 7, conv_args(t.a6, 64, B, H2, W2, t.a7, 64), kSrcPlain, kEpiPlain))) return rc;
  a = conv_args(t.a1, 32, B, H, W, t.a8, 32);
  a.xl = t.a7;
  a.cu = 64;
  if ((rc = fwd_fused(d, 8, a, kSrcUpCat, kEpiPlain))) return rc;
  if ((rc = fwd_fused(d, 9, conv_args(t.a8, 32, B, H, W, t.a9, 32), kSrcPlain, kEpiPlain))) return rc;
  a = conv_args(t.a9, 32, B, H, W, t.gm0, kLogitStride);
  a.kin = t.in32;
  a.inputs = d->inputs;
  a.target = t.tgt;
  a.inv_count = t.inv;
  a.err = d->err_sum;
  if ((rc = fwd_fused(d, 10, a, kSrcPlain, kEpiKpnLoss))) return rc;

  // the gradient through the ReLU of the layer whose output is act
  auto mask = [](const uint16_t* act, int ys, uint16_t* gm) {
    ConvArgs m{};
    m.act = act;
    m.ys = ys;
    m.y16 = gm;
    return m;
  };
  // through an upsample-and-concatenate: channels < cu to the low-resolution
  // layer (output act), the others to the skip's fp32 gradient
  auto upgrad = [](const uint16_t* act, int cu, uint16_t* gm, float* skip, int ss) {
    ConvArgs m{};
    m.act = act;
    m.cu = cu;
    m.y16 = gm;
    m.y32 = skip;
    m.ys = ss;
    return m;
  };
  auto poolgrad = [](const uint16_t* act, int ys, uint16_t* gm, const float* skip) {
    ConvArgs m{};
    m.act = act;
    m.ys = ys;
    m.y16 = gm;
    m.skip = skip;
    return m;
  };
  uint16_t *g0 = t.gm0, *g1 = t.gm1;
  if ((rc = bwd(d, 10, B, H, W, g0, t.a9, 32, nullptr, 0, mask(t.a9, 32, g1), kEpiMask))) return rc;
  if ((rc = bwd(d, 9, B, H, W, g1, t.a8, 32, nullptr, 0, mask(t.a8, 32, g0), kEpiMask))) return rc;
  if ((rc = bwd(d, 8, B, H, W, g0, t.a1, 32, t.a7, 64, upgrad(t.a7, 64, g1, t.skip1, 32), kEpiUpGrad))) return rc;
  if ((rc = bwd(d, 7, B, H2, W2, g1, t.a6, 64, nullptr, 0, mask(t.a6, 64, g0), kEpiMask))) return rc;
  if ((rc = bwd(d, 6, B, H2, W2, g0, t.a3, 64, t.a5, 96, upgrad(t.a5, 96, g1, t.skip3, 64), kEpiUpGrad))) return rc;
  if ((rc = bwd(d, 5, B, H4, W4, g1, t.a4, 96, nullptr, 0, mask(t.a4, 96, g0), kEpiMask))) return rc;
  if ((rc = bwd(d, 4, B, H4, W4, g0, t.p2, 64, nullptr, 0, poolgrad(t.a3, 64, g1, t.skip3), kEpiPoolGrad))) return rc;
  if ((rc = bwd(d, 3, B, H2, W2, g1, t.a2, 64, nullptr, 0, mask(t.a2, 64, g0), kEpiMask))) return rc;
  if ((rc = bwd(d, 2, B, H2, W2, g0, t.p1, 32, nullptr, 0, poolgrad(t.a1, 32, g1, t.skip1), kEpiPoolGrad))) return rc;
  if ((rc = bwd(d, 1, B, H, W, g1, t.a0, 32, nullptr, 0, mask(t.a0, 32, g0), kEpiMask))) return rc;
  return bwd(d, 0, B, H, W, g0, t.x0, d->in_pad, nullptr, 0, ConvArgs{}, -1);
}

// Loss gradient of `count` host pairs into grads and err_sum, in parts of as
// many images as the training buffers hold; pair i's squared error is weighted
// by inv * weights[i] (1 without weights).
int loss_gradient(mdwt_denoiser* d, const float* in, const float* tgt, const float* weights, int count,
                  float inv) {
  const size_t n = size_t(d->H) * d->W;
  int rc = train_bufs(d, count);
  if (rc) return rc;
  DNCHK(d, hipMemsetAsync(d->grads, 0, d->n_params * sizeof(float), d->stream));
  DNCHK(d, hipMemsetAsync(d->err_sum, 0, sizeof(float), d->stream));
  std::vector<float> w(size_t(std::min(count, d->train.images)));
  for (int i = 0; i < count; i += d->train.images) {
    const int B = std::min(count - i, d->train.images);
    for (int k = 0; k < B; ++k) w[size_t(k)] = weights ? inv * weights[i + k] : inv;
    DNCHK(d, hipMemcpyAsync(d->train.inv, w.data(), size_t(B) * sizeof(float), hipMemcpyHostToDevice, d->stream));
    DNCHK(d, mdwt::copy_to_device(d->train.in32, in + size_t(i) * n * d->inputs,
                                  size_t(B) * n * d->inputs * sizeof(float), d->device, d->stream));
    DNCHK(d, mdwt::copy_to_device(d->train.tgt, tgt + size_t(i) * n * 3, size_t(B) * n * 3 * sizeof(float),
                                  d->device, d->stream));
    if ((rc = train_batch(d, B))) return rc;
    DNCHK(d, hipStreamSynchronize(d->stream));  // the host's arrays are its own again
  }
  return MDWT_OK;
}

}  // namespace

extern "C" {

int mdwt_dn_create(mdwt_denoiser** out, int hip_device, int width, int height, int channels,
                   uint32_t seed) {
  if (!out) return MDWT_ERR_ARG;
  *out = nullptr;
  if (width < 4 || height < 4 || width % 4 || height % 4 || width > 8192 || height > 8192 ||
      channels < 1 || channels > 12)
    return MDWT_ERR_ARG;
  // The element-wise kernels index pixel x channel in 32-bit ints; the widest
  // full-resolution tensor has 96 channels (the level-0 concatenation), so
  // 2^24 pixels keep every index below 2^31.
  if (size_t(width) * size_t(height) > kMaxPixels) return MDWT_ERR_LIMIT;
  auto* d = new (std::nothrow) mdwt_denoiser();
  if (!d) return MDWT_ERR_OOM;
  mdwt::host_copy_acquire();
  d->device = hip_device;
  d->W = width;
  d->H = height;
  d->channels = channels;
  d->inputs = mdwt::dn::input_width(channels);
  d->in_pad = round_up(d->inputs, 8);
  int rc = MDWT_OK;
  if (hipSetDevice(hip_device) != hipSuccess ||
      hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&d->ev0) != hipSuccess || hipEventCreate(&d->ev1) != hipSuccess)
    rc = MDWT_ERR_HIP;
  if (rc == MDWT_OK) rc = setup(d, seed);
  if (rc == MDWT_OK) rc = refresh_weights(d);
  if (rc == MDWT_OK && hipStreamSynchronize(d->stream) != hipSuccess) rc = MDWT_ERR_HIP;
  if (rc != MDWT_OK) {
    mdwt_dn_destroy(d);
    return rc;
  }
  *out = d;
  return MDWT_OK;
}

int mdwt_dn_destroy(mdwt_denoiser* d) {
  if (!d) return MDWT_ERR_ARG;
  (void)hipSetDevice(d->device);
  if (d->stream) (void)hipStreamSynchronize(d->stream);
  free_train(&d->train);
  for (void* p : d->bufs) (void)hipFree(p);
  if (d->ev0) (void)hipEventDestroy(d->ev0);
  if (d->ev1) (void)hipEventDestroy(d->ev1);
  if (d->stream) (void)hipStreamDestroy(d->stream);
  mdwt::host_copy_release();
  delete d;
  return MDWT_OK;
}

const char* mdwt_dn_last_error(const mdwt_denoiser* d) { return d ? d->err.c_str() : ""; }

int mdwt_dn_num_params(const mdwt_denoiser* d, int* n) {
  if (!d || !n) return MDWT_ERR_ARG;
  *n = int(d->n_params);
  return MDWT_OK;
}

int mdwt_dn_get_params(mdwt_denoiser* d, float* out) {
  if (!d || !out) return MDWT_ERR_ARG;
  DNCHK(d, hipSetDevice(d->device));
  DNCHK(d, hipStreamSynchronize(d->stream));
  DNCHK(d, mdwt::copy_to_host(out, d->params, d->n_params * sizeof(float), d->device, d->stream));
  return MDWT_OK;
}

int mdwt_dn_set_params(mdwt_denoiser* d, const float* in) {
  if (!d || !in) return MDWT_ERR_ARG;
  DNCHK(d, hipSetDevice(d->device));
  DNCHK(d, hipStreamSynchronize(d->stream));
  DNCHK(d, hipMemcpy(d->params, in, d->n_params * sizeof(float), hipMemcpyHostToDevice));
  int rc = refresh_weights(d);
  if (rc) return rc;
  DNCHK(d, hipStreamSynchronize(d->stream));
  return MDWT_OK;
}

int mdwt_dn_infer(mdwt_denoiser* d, const float* input, float* output, float* ms) {
  if (!d || !input || !output) return MDWT_ERR_ARG;
  DNCHK(d, hipSetDevice(d->device));
  const size_t n = size_t(d->H) * d->W;
  DNCHK(d, mdwt::copy_to_device(d->in32, input, n * d->inputs * sizeof(float), d->device, d->stream));
  DNCHK(d, hipEventRecord(d->ev0, d->stream));
  int rc = d->fused ? forward_fused(d) : forward(d);
  if (rc) return rc;
  DNCHK(d, hipEventRecord(d->ev1, d->stream));
  DNCHK(d, mdwt::copy_to_host(output, d->pred, n * 3 * sizeof(float), d->device, d->stream));
  DNCHK(d, hipStreamSynchronize(d->stream));
  float t = 0.f;
  DNCHK(d, hipEventElapsedTime(&t, d->ev0, d->ev1));
  if (ms) *ms = t;
  return MDWT_OK;
}

int mdwt_dn_set_fused(mdwt_denoiser* d, int on) {
  if (!d) return MDWT_ERR_ARG;
  d->fused = on != 0;
  return MDWT_OK;
}

int mdwt_dn_gradient(mdwt_denoiser* d, const float* input, const float* target, float* grad,
                     float* loss) {
  if (!d || !input || !target || !grad) return MDWT_ERR_ARG;
  DNCHK(d, hipSetDevice(d->device));
  const size_t n = size_t(d->H) * d->W;
  int rc = loss_gradient(d, input, target, nullptr, 1, 1.f / float(n * 3));
  if (rc) return rc;
  DNCHK(d, mdwt::copy_to_host(grad, d->grads, d->n_params * sizeof(float), d->device, d->stream));
  if (loss) {
    float e = 0.f;
    DNCHK(d, hipMemcpy(&e, d->err_sum, sizeof(float), hipMemcpyDeviceToHost));
    *loss = e / float(n * 3);
  }
  return MDWT_OK;
}

int mdwt_dn_train_step(mdwt_denoiser* d, const float* inputs, const float* targets,
                       const float* weights, int count, float lr, float* loss) {
  if (!d || !inputs || !targets || count < 1 || !(lr > 0.f)) return MDWT_ERR_ARG;
  for (int i = 0; weights && i < count; ++i)
    if (!(weights[i] >= 0.f) || std::isinf(weights[i])) return MDWT_ERR_ARG;
  DNCHK(d, hipSetDevice(d->device));
  const size_t n = size_t(d->H) * d->W;
  const float inv = 1.f / float(n * 3 * size_t(count));
  int rc = loss_gradient(d, inputs, targets, weights, count, inv);
  if (rc) return rc;
  ++d->step;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - std::pow(b1, float(d->step)), c2 = 1.f - std::pow(b2, float(d->step));
  DNCHK(d, mdwt::dn::adam(d->params, d->grads, d->mom, d->var, int(d->n_params), lr, b1, b2, c1, c2, eps,
                          d->stream));
  rc = refresh_weights(d);
  if (rc) return rc;
  float e = 0.f;
  DNCHK(d, hipMemcpyAsync(&e, d->err_sum, sizeof(float), hipMemcpyDeviceToHost, d->stream));
  DNCHK(d, hipStreamSynchronize(d->stream));
  if (loss) *loss = e / float(n * 3 * size_t(count));
  return MDWT_OK;
}

}  // extern "C"
