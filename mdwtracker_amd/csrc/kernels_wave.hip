// Wave-coherent frame kernels (schedule 1) without lighting: instantiations of
// wave_paths.hpp for one view and for batched views, and their selection.
#include "wave_paths.hpp"

namespace mdwt {
namespace {

// form: 0 one view, 1 batched views (one launch), 2 batched views (persistent),
// 3 one view, several frames
template <int MODE, int DT, bool WIDE>
RenderFn wave_fn_form(int form) {
  switch (form) {
    case 0: return render_wave<MODE, DT, WIDE, false>;
    case 1: return render_views_wave<MODE, DT, WIDE, false>;
    case 2: return render_views_wave_persistent<MODE, DT, WIDE>;
    default: return render_wave_team<MODE, DT, WIDE, false>;
  }
}
template <int MODE, bool WIDE>
RenderFn wave_fn(int dtype, int form) {
  switch (dtype) {
    case MDWT_DT_U8: return wave_fn_form<MODE, MDWT_DT_U8, WIDE>(form);
    case MDWT_DT_U16: return wave_fn_form<MODE, MDWT_DT_U16, WIDE>(form);
    case MDWT_DT_F16: return wave_fn_form<MODE, MDWT_DT_F16, WIDE>(form);
    default: return wave_fn_form<MODE, MDWT_DT_F32, WIDE>(form);
  }
}

}  // namespace

bool wave_schedule_applies(const RenderParams& p, int mode, bool count) {
  // a ray visits at most mx + my + mz cells: visit numbers fit the records' 26 bits
  const uint64_t max_visits = uint64_t(p.mc[0]) + uint64_t(p.mc[1]) + uint64_t(p.mc[2]);
  return mode >= 0 && mode <= 5 && !count && p.vol.channels <= kMaxChannels &&
         max_visits < (uint64_t(1) << kVisitBits);
}

RenderFn select_wave_kernel(const RenderParams& p, int mode, int dtype, int form) {
  if (is_shaded(p)) return select_wave_lit_kernel(p, mode, dtype, form);
  if (mode == 0)
    return p.vol.channels > 4 ? wave_fn<0, true>(dtype, form) : wave_fn<0, false>(dtype, form);
  if (mode == 3)
    return p.vol.channels > 4 ? wave_fn<3, true>(dtype, form) : wave_fn<3, false>(dtype, form);
  if (mode == 4)
    return p.vol.channels > 4 ? wave_fn<4, true>(dtype, form) : wave_fn<4, false>(dtype, form);
  if (mode == 5)
    return p.vol.channels > 4 ? wave_fn<5, true>(dtype, form) : wave_fn<5, false>(dtype, form);
  if (mode == 1)
    return p.vol.channels > 4 ? wave_fn<1, true>(dtype, form) : wave_fn<1, false>(dtype, form);
  return p.vol.channels > 4 ? wave_fn<2, true>(dtype, form) : wave_fn<2, false>(dtype, form);
}

size_t wave_lds_bytes(const RenderParams& p) {
  static_assert(sizeof(WaveLds<kRecords>) % 16 == 0 && sizeof(WaveLds<kRecordsWide>) % 16 == 0,
                "the opacity table follows the per-wave LDS");
  return size_t(p.vol.channels) * size_t(p.tf.stride) * sizeof(float);
}

}  // namespace mdwt
