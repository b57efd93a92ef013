"""Volumes whose copies pass 4 GiB, where the samplers use 64-bit addresses: four
f32 channels of 650^3 voxels (bricks and joint copy of 4.4 GB each) against the
same values as f16 (2.2 GB each, 32-bit addresses): the same images."""
import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu

N = 650


@pytest.fixture(scope="module")
def capi():
    from mdwtracker_amd import capi
    return capi


@pytest.fixture(scope="module")
def volume():
    """f16 values, so that both types hold them exactly."""
    rng = np.random.default_rng(8)
    v = scenes.normalise(scenes.noise_blob_volume((50, 50, 50), 6, rng)).astype(np.float32)
    v = np.tile(v, (N // 50,) * 3)
    # so that no two layers, rows or columns are the same
    v *= np.linspace(0.6, 1.0, N, dtype=np.float32)
    v *= np.linspace(1.0, 0.7, N, dtype=np.float32)[:, None]
    v *= np.linspace(0.8, 1.0, N, dtype=np.float32)[:, None, None]
    return v.astype(np.float16)


def _images(capi, volume):
    """-m 0 to 2, the gradient shading and -m 9 sample the bricks, the others the
    joint copy; one frame, then several per launch."""
    r = capi.MdwtRenderer(0)
    rng = np.random.default_rng(2)
    for _ in range(4):
        r.push_channel(volume)
    r.init(2, (26, 26, 26), False)
    for c in range(4):
        r.set_tf(c, scenes.piecewise_tf(6, rng, 0.25 * c, x_lo=0.2, clear_first=True), 0.02, (0.0, 1.0))
    r.set_frame(96, 80, 1, True, (0.1, 0.2, 0.3))
    r.set_seed(4)
    out = []
    for mode, schedule, shaded in ((2, 1, False), (2, 1, True), (1, 0, False), (3, 1, False), (5, 1, True),
                                   (4, 0, False), (8, 1, False), (9, 1, False)):
        print(f"[large] {volume.dtype} mode {mode} schedule {schedule} shaded {shaded}", flush=True)
        r.set_mode(mode)
        r.set_schedule(schedule)
        r.set_light((0.3, -1.0, 0.2), shaded, shaded)
        for cam in (scenes.orbit_camera(1.6), ((0.5, 0.5, 2.2), (0.5, 0.5, 0.5), (0.0, 1.0, 0.0), 40.0)):
            r.set_camera(*cam)
            r.reset_accumulation()
            for n in (1, 4):
                r.render(n)
                out.append(r.read_accum())
    r.close()
    return out


def test_64_bit_addresses(capi, volume):
    small = _images(capi, volume)
    large = _images(capi, volume.astype(np.float32))
    for k, (a, b) in enumerate(zip(small, large)):
        assert a[..., :3].std() > 0.01, k
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32), err_msg=str(k))
