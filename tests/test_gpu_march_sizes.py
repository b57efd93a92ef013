"""One frame of the ray marchers around the frame sizes at which another instance
of their kernel takes over (2-byte voxels: two or three waves per SIMD), against
the several-frame kernel."""
import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu


# pixel blocks of 256: 512 and 528 (two waves per SIMD: 512, with shading), 768 and
# 792 (three: 768), and the same in blocks of 64
@pytest.mark.parametrize("size,block", [((512, 256), 256), ((528, 256), 256), ((512, 384), 256), ((528, 384), 256),
                                        ((512, 384), 64), ((520, 384), 64)])
@pytest.mark.parametrize("mode,dtype,lit", [(6, np.uint16, True), (7, np.float16, False), (8, np.float16, True),
                                            (8, np.uint16, False), (8, np.uint8, True), (8, np.float32, True)])
def test_one_frame_at_the_instances_sizes(mode, dtype, lit, size, block):
    from mdwtracker_amd import capi
    out = []
    for split in (False, True):
        print(f"[march] mode {mode} {np.dtype(dtype)} lit {lit} {size} block {block} split {split}", flush=True)
        rng = np.random.default_rng(6)
        r = capi.MdwtRenderer(0)
        for _ in range(3):
            v = scenes.normalise(scenes.noise_blob_volume((17, 22, 19), 6, rng))
            top = np.iinfo(dtype).max if np.issubdtype(dtype, np.integer) else 1
            r.push_channel((np.rint(v * top) if top > 1 else v).astype(dtype))
        r.init(mode, (4, 5, 3), False)
        for c in range(3):
            r.set_tf(c, scenes.piecewise_tf(6, rng, c / 3, x_lo=0.2, clear_first=True), 0.2, (0.0, 1.0))
        r.set_block(block)
        r.set_frame(size[0], size[1], 1, True, (0.1, 0.2, 0.3))
        r.set_light((0.3, -1.0, 0.2), lit, lit)
        r.set_camera(*scenes.orbit_camera(1.6))
        for _ in range(4 if split else 1):
            r.render(1 if split else 4)
        out.append(r.read_accum().view(np.uint32))
        r.close()
    np.testing.assert_array_equal(*out)
