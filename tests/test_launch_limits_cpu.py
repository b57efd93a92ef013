"""Which launches the dispatch chooses at the limits of its arguments, checked
on the host: a program linked against libmdwt.so asks the library's own rules."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "mdwtracker_amd"

PROLOGUE = r"""
#include <cstdio>
#include <cstring>
#include "mdwt_internal.hpp"
using namespace mdwt;
static int bad = 0;
#define EXPECT(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); ++bad; } } while (0)
static RenderParams params(int blocks, int items, int bw, int bh) {
  RenderParams p;
  std::memset(&p, 0, sizeof(p));
  p.vol.channels = 4;
  p.tf.stride = 64;
  for (int& m : p.mc) m = 8;
  p.fr.schedule = 1;
  p.fr.n_blocks = blocks;
  p.fr.n_items = items;
  p.fr.bw = bw;
  p.fr.bh = bh;
  return p;
}
"""


def run(tmp_path, body):
    if not (PKG / "libmdwt.so").exists():
        pytest.skip("libmdwt.so is not built")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROLOGUE + "int main() {\n" + body + '\n  if (!bad) std::printf("ok\\n");\n  return bad;\n}\n')
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        f"-I{ROOT / 'include'}", f"-I{PKG / 'csrc'}", str(src), str(PKG / "libmdwt.so"),
                        f"-Wl,-rpath,{PKG}", "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64",
                        "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_several_frames_only_where_the_grid_fits(tmp_path):
    """A workgroup of 256 threads per 8x8 pixels: HIP takes fewer than 2^32
    threads, so frames of 2^30 pixels and batches of as many go frame by frame
    (one thread per pixel), the next smaller ones several frames at a time."""
    run(tmp_path, r"""
  const struct { int bw, bh; } shapes[] = {{8, 8}, {16, 8}, {16, 16}};
  for (const auto& s : shapes) {
    const int q = s.bw * s.bh / 64, limit = (1 << 24) / q;  // blocks of 2^30 pixels
    for (int mode = 0; mode < 10; ++mode) {
      EXPECT(!several_frames_apply(params(limit, 0, s.bw, s.bh), mode, false));
      EXPECT(several_frames_apply(params(limit - 1, 0, s.bw, s.bh), mode, false));
      EXPECT(!several_frames_apply(params(1, 0, s.bw, s.bh), mode, true));  // the counting pass
      EXPECT(!several_view_frames_apply(params(0, limit, s.bw, s.bh), mode));
      EXPECT(!several_view_frames_apply(params(0, 2 * limit, s.bw, s.bh), mode));
      EXPECT(several_view_frames_apply(params(0, limit - 1, s.bw, s.bh), mode) == (mode <= 5));
    }
  }""")


def test_draws_of_a_launch_fit_32_bits(tmp_path):
    """Any sample count: whole rounds of four draws, at least one round or about
    32 draws, and never more draws than the kernels' 32-bit count holds."""
    run(tmp_path, r"""
  for (int64_t spp : {1ll, 2ll, 3ll, 4ll, 5ll, 6ll, 8ll, 31ll, 32ll, 33ll, 1000ll, (1ll << 28) - 1, 1ll << 28,
                      (1ll << 29) + 1, (1ll << 30) - 2, (1ll << 30) + 1, (1ll << 31) - 4, (1ll << 31) - 1})
    for (int left : {0, 1, 2, 3, 4, 5, 7, 32, 33, 100, 2147483647}) {
      const int64_t n = frames_per_launch(left, int(spp));
      EXPECT(n >= 0 && n <= left && n * spp % 4 == 0 && n * spp < (1ll << 31));
      EXPECT(n * spp <= 32 || n <= 4);
      if (left >= 4 && spp <= 1000) EXPECT(n > 0);
    }""")


def test_auxiliary_buffers_are_packed_in_pieces_that_fit(tmp_path):
    """A thread per value of a piece, for every channel count; the launcher takes
    no larger piece (a frame of 2^30 pixels has up to 14 values each)."""
    run(tmp_path, r"""
  for (int c = 1; c <= kMaxChannels; ++c) {
    const size_t n = pack_aov_pixels(2 + c);
    EXPECT(n > 0 && grid_fits((n * (2 + c) + 255) / 256, 256));
    const int row = 4 * aov_groups(c);
    EXPECT(launch_pack_aov(nullptr, row, 2 + c, n + 1, nullptr, nullptr) == hipErrorInvalidValue);
    EXPECT(launch_pack_aov(nullptr, row, 2 + c, size_t(1) << 30, nullptr, nullptr) == hipErrorInvalidValue);
  }""")


def test_persistent_grid_belongs_to_the_kernel(tmp_path):
    """The resident grid of launch form 2 is kept for one kernel: whatever changes
    the kernel, its tables or its workgroup (the schedule too) is another."""
    run(tmp_path, r"""
  for (int mode = 0; mode < 10; ++mode)
    for (int dtype = 0; dtype < 4; ++dtype) {
      RenderParams a = params(0, 100, 16, 16), b = a;
      const PersistentKernel k = persistent_kernel(a, mode, dtype);
      EXPECT(k.fn && k == persistent_kernel(b, mode, dtype));
      b.fr.schedule = 0;
      EXPECT((k == persistent_kernel(b, mode, dtype)) == (mode > 5));
      b = a;
      b.fr.sh.shadows = 1;
      EXPECT(!(k == persistent_kernel(b, mode, dtype)) || mode == 9);
      b = a;
      b.fr.bh = 8;
      EXPECT(!(k == persistent_kernel(b, mode, dtype)));
      b = a;
      b.tf.stride = 128;
      EXPECT(!(k == persistent_kernel(b, mode, dtype)));
      EXPECT(!(k == persistent_kernel(a, (mode + 1) % 10, dtype)));
      EXPECT(!(k == persistent_kernel(a, mode, (dtype + 1) % 4)));
    }""")


def test_no_kernel_for_a_form_that_has_none(tmp_path):
    """The persistent form has no shaded instance, and there are four forms; what
    has no kernel is not launched."""
    run(tmp_path, r"""
  for (int mode = 0; mode < 6; ++mode)
    for (int dtype = 0; dtype < 4; ++dtype)
      for (int channels : {4, 10})
        for (int shaded = 0; shaded < 2; ++shaded) {
          RenderParams p = params(1, 1, 16, 16);
          p.vol.channels = channels;
          p.fr.sh.gradient = shaded;
          RenderFn seen[4];
          for (int form = 0; form < 4; ++form) {
            seen[form] = select_wave_kernel(p, mode, dtype, form);
            EXPECT((seen[form] != nullptr) == !(shaded && form == 2));
            for (int k = 0; k < form; ++k) EXPECT(seen[form] != seen[k]);
          }
          EXPECT(!select_wave_kernel(p, mode, dtype, -1) && !select_wave_kernel(p, mode, dtype, 4));
          EXPECT(persistent_kernel(p, mode, dtype).fn);
        }
  PersistentKernel none;
  int n = 0;
  EXPECT(persistent_blocks_per_cu(none, &n) == hipErrorInvalidValue);""")
