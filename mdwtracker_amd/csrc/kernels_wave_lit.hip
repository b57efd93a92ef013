// Wave-coherent frame kernels (schedule 1) with gradient shading and shadow
// rays: instantiations of wave_paths.hpp for one view and for batched views in
// one launch, and their selection. Beside the plain kernels (whose registers
// and code they would cost), in a source of their own for build time.
// A hit's six gradient samples and its shadow ray's rounds run in the wave that
// traced it, so a shadow ray's steps are compacted like a camera ray's: at
// 1024^2 on four 256^3 u8 channels with both (-m 2), a frame was 745 us on the
// thread-per-pixel kernel (23% of lanes active) and is about 250 us here. The
// denoiser's buffers need no instance of their own: a wave writes them after
// the sample is composited (64 frames of 512^2: 9.2 -> 3.6 ms; plain frames
// unchanged).
#include "wave_paths.hpp"

namespace mdwt {
namespace {

template <int MODE, int DT, bool WIDE>
RenderFn lit_fn_form(int form) {
  switch (form) {
    case 0: return render_wave<MODE, DT, WIDE, true>;
    case 1: return render_views_wave<MODE, DT, WIDE, true>;
    default: return render_wave_team<MODE, DT, WIDE, true>;
  }
}
template <int MODE, bool WIDE>
RenderFn lit_fn(int dtype, int form) {
  switch (dtype) {
    case MDWT_DT_U8: return lit_fn_form<MODE, MDWT_DT_U8, WIDE>(form);
    case MDWT_DT_U16: return lit_fn_form<MODE, MDWT_DT_U16, WIDE>(form);
    case MDWT_DT_F16: return lit_fn_form<MODE, MDWT_DT_F16, WIDE>(form);
    default: return lit_fn_form<MODE, MDWT_DT_F32, WIDE>(form);
  }
}

}  // namespace

RenderFn select_wave_lit_kernel(const RenderParams& p, int mode, int dtype, int form) {
  const bool wide = p.vol.channels > 4;
  switch (mode) {
    case 0: return wide ? lit_fn<0, true>(dtype, form) : lit_fn<0, false>(dtype, form);
    case 1: return wide ? lit_fn<1, true>(dtype, form) : lit_fn<1, false>(dtype, form);
    case 2: return wide ? lit_fn<2, true>(dtype, form) : lit_fn<2, false>(dtype, form);
    case 3: return wide ? lit_fn<3, true>(dtype, form) : lit_fn<3, false>(dtype, form);
    case 4: return wide ? lit_fn<4, true>(dtype, form) : lit_fn<4, false>(dtype, form);
    default: return wide ? lit_fn<5, true>(dtype, form) : lit_fn<5, false>(dtype, form);
  }
}

}  // namespace mdwt
