// Host-side launchers of the MDWT kernels (defined in the .hip files, called
// by the C ABI in mdwt_api.cpp). Each returns the launch status.
#pragma once
#include <hip/hip_runtime.h>

#include "mdwt_types.hpp"

namespace mdwt {

// host stub of a frame kernel
using RenderFn = void (*)(RenderParams);
// gradient shading or shadow rays
inline bool is_shaded(const RenderParams& p) { return p.fr.sh.shadows != 0 || p.fr.sh.gradient != 0; }
// wave-coherent frame kernels (kernels_wave.hip, and kernels_wave_lit.hip with
// shading; schedule 1): -m 0 to -m 5 on at most twelve channels, not the
// counting pass; form 0 one view, 1 batched views in one launch, 2 batched
// views in a persistent launch (not with shading), 3 p.fr.team_frames frames of
// one view in one launch
bool wave_schedule_applies(const RenderParams& p, int mode, bool count);
RenderFn select_wave_kernel(const RenderParams& p, int mode, int dtype, int form);
// whether HIP takes a launch of `blocks` workgroups of `threads` threads along x:
// it supports fewer than 2^32 threads. The several-frame kernels have a
// workgroup of 256 threads per 64 pixels, four times the one-frame kernels'
// threads, and pass it at 2^30 pixels.
inline bool grid_fits(uint64_t blocks, uint64_t threads) { return blocks * threads < (uint64_t(1) << 32); }
// whether launch_render can render several frames (team_frames) in one launch:
// the wave-coherent modes and the ray marchers, where the grid fits
bool several_frames_apply(const RenderParams& p, int mode, bool count);
// Frames of a several-frame launch when `left` are to be rendered, or 0 for one
// frame by the one-frame kernels. The team kernel's four waves take four draws
// (samples) at a time: only whole rounds of four draws, since in a partial one
// waves hold their workgroup's LDS and do nothing. About 32 draws: longer
// launches gained under 1 %. The draws of a launch stay below 2^30 (the kernel
// counts them in 32 bits).
constexpr int kTeamDraws = 32;
inline int frames_per_launch(int left, int spp) {
  if (spp >= 1 << 28) return 0;
  const int step = spp % 4 == 0 ? 1 : (spp % 2 == 0 ? 2 : 4), most = kTeamDraws / spp;
  const int n = most > step ? most : step;
  return (left < n ? left : n) / step * step;
}
// the same of launch_views: the wave-coherent modes, where the grid fits
bool several_view_frames_apply(const RenderParams& p, int mode);
// its parts: shaded -m 0 / 1 / 2, and -m 3 / 4 / 5 plain and shaded
RenderFn select_wave_lit_kernel(const RenderParams& p, int mode, int dtype, int form);
RenderFn select_wave_sum_kernel(const RenderParams& p, int mode, int dtype, int form);
RenderFn select_wave_lit_sum_kernel(const RenderParams& p, int mode, int dtype, int form);
// dynamic LDS of a wave-coherent launch (transfer-function opacities)
size_t wave_lds_bytes(const RenderParams& p);

hipError_t launch_ranges(const RangeParams& p, int dtype, hipStream_t s);
hipError_t launch_majorants(const MajorantParams& p, hipStream_t s);
// order (nb blocks) by decreasing cost, block b's being the sum of ticks[wpb * b ..]
// (the block at position b); tmp: nb entries
hipError_t launch_cost_order(uint32_t* order, const uint32_t* ticks, uint32_t* tmp, int nb, int wpb,
                             hipStream_t s);
// out[p][0 .. nv) = aov[p][0 .. nv) of rows of `row` floats, n pixels: at most
// pack_aov_pixels(nv), 64 MiB of output (a thread per value stays far below the
// threads that HIP takes, and the scratch small beside the image)
inline size_t pack_aov_pixels(int nv) { return (size_t(64) << 20) / (size_t(nv) * sizeof(float)); }
hipError_t launch_pack_aov(const float* aov, int row, int nv, size_t n, float* out, hipStream_t s);
// v.bricks (brick_stride bytes per channel) = v.vol in 4 x 4 x 4 bricks
hipError_t launch_bricks(const VolumeParams& v, int dtype, hipStream_t s);
// v.joint (joint_stride bytes per group of four channels) from v.vol
hipError_t launch_joint(const VolumeParams& v, int dtype, hipStream_t s);
hipError_t launch_render(const RenderParams& p, int mode, int dtype, bool count, hipStream_t s);
// batched views, launch form 2: the persistent frame kernel over p.fr.items
// (grid workgroups, workgroup g takes items g, g + grid, ...) at the ids in
// p.fr.work[1..2], then the kernel that advances those ids; the pair is what a
// graph captures for one frame
hipError_t launch_views_persistent(const RenderParams& p, int mode, int dtype, int grid,
                                   hipStream_t s);
// the kernel that it launches for p (the schedule, mode, shading, channels and
// block shape choose it), and its resident workgroups per CU
struct PersistentKernel {
  RenderFn fn = nullptr;
  size_t lds = 0;
  int threads = 0;
  bool operator==(const PersistentKernel& o) const {
    return fn == o.fn && lds == o.lds && threads == o.threads;
  }
};
PersistentKernel persistent_kernel(const RenderParams& p, int mode, int dtype);
hipError_t persistent_blocks_per_cu(const PersistentKernel& k, int* out);
// batched views in one launch: one workgroup per item of p.fr.items (view,
// pixel block), frame and accumulation ids from p.fr.frame_id / accum_id
hipError_t launch_views(const RenderParams& p, int mode, int dtype, bool count, hipStream_t s);
// dynamic LDS of a frame launch (transfer-function texels)
size_t render_lds_bytes(const RenderParams& p);
hipError_t launch_gen_rays(const CameraParams& cam, int W, int H, uint32_t seed, uint32_t frame,
                           uint32_t sample, int jitter2d, float* org, float* dir, hipStream_t s);
hipError_t launch_clip(const VolumeParams& vol, const float* org, const float* dir, int n,
                       float* t01, int* hit, hipStream_t s);
hipError_t launch_trace_cells(const VolumeParams& vol, const int mc[3], const float* org,
                              const float* dir, int n, int max_cells, int* cells, float* t01,
                              int* counts, hipStream_t s);
hipError_t launch_rgba8(const void* accum, uint32_t* out, int n, hipStream_t s);
// Allocation-free frame-buffer read: a file-scope device array of
// kFbScratchPixels RGBA8 pixels per GPU. fb_scratch_setup (once per device,
// with that device current; called by mdwt_init) takes its address with
// hipGetSymbolAddress; fb_scratch returns it (nullptr before the set-up).
constexpr size_t kFbScratchPixels = size_t(1) << 20;
hipError_t fb_scratch_setup(int device);
uint32_t* fb_scratch(int device);
hipError_t launch_copy(const void* src, void* dst, size_t n16, hipStream_t s);
// read-only reduction over n16 float4 (bandwidth probe): kReadGrid workgroups,
// one partial sum each into sums
constexpr unsigned kReadGrid = 4096;
hipError_t launch_read(const void* src, size_t n16, float* sums, hipStream_t s);

}  // namespace mdwt
