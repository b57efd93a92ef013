// Wave-coherent frame kernels (schedule 1) of -m 0 / 1 / 2 without lighting:
// instantiations of wave_paths.hpp for one view and for batched views, and the
// selection among all of them.
#include "wave_paths.hpp"

namespace mdwt {

bool wave_schedule_applies(const RenderParams& p, int mode, bool count) {
  // a ray visits at most mx + my + mz cells: visit numbers fit the records' 26 bits
  const uint64_t max_visits = uint64_t(p.mc[0]) + uint64_t(p.mc[1]) + uint64_t(p.mc[2]);
  return mode >= 0 && mode <= 5 && !count && p.vol.channels <= kMaxChannels &&
         max_visits < (uint64_t(1) << kVisitBits);
}

RenderFn select_wave_kernel(const RenderParams& p, int mode, int dtype, int form) {
  const bool lit = is_shaded(p);
  if (mode >= 3) return lit ? select_wave_lit_sum_kernel(p, mode, dtype, form)
                            : select_wave_sum_kernel(p, mode, dtype, form);
  if (lit) return select_wave_lit_kernel(p, mode, dtype, form);
  if (mode == 0) return wave_fn<0, false>(p, dtype, form);
  return mode == 1 ? wave_fn<1, false>(p, dtype, form) : wave_fn<2, false>(p, dtype, form);
}

size_t wave_lds_bytes(const RenderParams& p) {
  static_assert(sizeof(WaveLds<kRecords>) % 16 == 0 && sizeof(WaveLds<kRecordsWide>) % 16 == 0,
                "the opacity table follows the per-wave LDS");
  return size_t(p.vol.channels) * size_t(p.tf.stride) * sizeof(float);
}

}  // namespace mdwt
