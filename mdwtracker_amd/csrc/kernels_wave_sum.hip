// Wave-coherent kernels of the modes that track the summed majorant (-m 3 / 4 / 5),
// plain (wave_paths.hpp). A file of its own: the instances take minutes to compile.
#include "wave_paths.hpp"

namespace mdwt {

RenderFn select_wave_sum_kernel(const RenderParams& p, int mode, int dtype, int form) {
  if (mode == 3) return wave_fn<3, false>(p, dtype, form);
  return mode == 4 ? wave_fn<4, false>(p, dtype, form) : wave_fn<5, false>(p, dtype, form);
}

}  // namespace mdwt
