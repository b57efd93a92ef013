// Wave-coherent frame kernels (schedule 1) of -m 0 / 1 / 2 with gradient shading and
// shadow rays: instantiations of wave_paths.hpp for one view and for batched views
// in one launch. Beside the plain kernels (whose registers
// and code they would cost), in a source of their own for build time.
// A hit's six gradient samples and its shadow ray's rounds run in the wave that
// traced it, so a shadow ray's steps are compacted like a camera ray's: at
// 1024^2 on four 256^3 u8 channels with both (-m 2), a frame was 745 us on the
// thread-per-pixel kernel (23% of lanes active) and is about 250 us here. The
// denoiser's buffers need no instance of their own: a wave writes them after
// the sample is composited (64 frames of 512^2: 9.9 -> 4.4 ms; plain frames
// unchanged).
#include "wave_paths.hpp"

namespace mdwt {

RenderFn select_wave_lit_kernel(const RenderParams& p, int mode, int dtype, int form) {
  if (mode == 0) return wave_fn<0, true>(p, dtype, form);
  return mode == 1 ? wave_fn<1, true>(p, dtype, form) : wave_fn<2, true>(p, dtype, form);
}

}  // namespace mdwt
