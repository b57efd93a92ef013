"""The default frame kernels against the thread-per-pixel schedule (itself
bit-exact against the oracle, test_gpu_parity.py): identical images, second
moments and auxiliary buffers at the sizes and options where the paths differ."""
import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from mdwtracker_amd import capi
    return capi


def volume(channels, dtype, dims=(37, 29, 42), seed=5):
    """(channel volumes (nz, ny, nx), transfer functions) of a small ragged scene."""
    rng = np.random.default_rng(seed)
    vols, tfs = [], []
    for c in range(channels):
        v = scenes.normalise(scenes.noise_blob_volume(dims[::-1], 6, rng))
        vols.append(scenes.quantize_u8(v) if dtype == np.uint8 else
                    np.rint(v * 65535).astype(np.uint16) if dtype == np.uint16 else v.astype(dtype))
        tfs.append(scenes.piecewise_tf(6, rng, c / channels, x_lo=0.2, clear_first=True))
    return vols, tfs


def renderer(capi, vols, tfs, mode, size, spp, schedule, mc=(5, 4, 6), opacity=0.08):
    r = capi.MdwtRenderer(0)
    for v in vols:
        r.push_channel(v)
    r.init(mode, mc, False)
    r.set_schedule(schedule)
    for c, t in enumerate(tfs):
        r.set_tf(c, t, opacity, (0.0, 1.0))
    r.set_frame(size[0], size[1], spp, True, (0.1, 0.2, 0.3))
    r.set_camera(*scenes.orbit_camera(1.6))
    r.set_seed(11)
    return r


@pytest.mark.parametrize("channels,dtype", [(1, np.uint16), (3, np.uint8), (10, np.float32)])
@pytest.mark.parametrize("mode", [0, 1, 2, 3, 4, 5])
def test_shading_and_aov_on_both_schedules(capi, mode, channels, dtype):
    """Gradient shading, shadow rays and the denoiser's buffers, alone and
    together, on a frame whose sides are not multiples of 8."""
    vols, tfs = volume(channels, dtype)
    for shadows, gradient, aov in ((1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1)):
        out = []
        for schedule in (0, 1):
            print(f"[paths] mode {mode} channels {channels} shadows {shadows} gradient {gradient} "
                  f"aov {aov} schedule {schedule}", flush=True)
            r = renderer(capi, vols, tfs, mode, (75, 51), 2, schedule)
            r.set_light((0.3, -1.0, 0.2), bool(shadows), bool(gradient))
            r.set_moments(True)
            r.set_aov(bool(aov))
            r.set_aov_frames(2)
            r.render(3)
            got = list(r.read_accum(with_m2=True)) + ([r.read_aov()] if aov else [])
            assert got[0][..., :3].std() > 0.01
            out.append([g.view(np.uint32) for g in got])
            r.close()
        for a, b in zip(*out):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("mode,channels,dtype,shaded", [
    (0, 3, np.uint8, False), (0, 5, np.uint16, False), (1, 4, np.float16, False),
    (2, 4, np.uint8, False), (2, 10, np.float32, True), (3, 2, np.uint16, True),
    (4, 4, np.uint8, False), (5, 1, np.float32, True), (6, 2, np.uint16, False),
    (7, 3, np.uint8, True), (8, 4, np.float32, False), (9, 5, np.float16, True)])
def test_several_frames_in_one_launch(capi, mode, channels, dtype, shaded):
    """n frames in one call against n calls of one frame: around the launch's
    rounds of four draws and its 32 draws, with the auxiliary buffers ending
    inside the call, with and without accumulation, small workgroups."""
    vols, tfs = volume(channels, dtype)
    for size, spp, frames, accumulate, aov, block in (
            ((9, 7), 1, 4, True, 0, 256), ((75, 51), 1, 39, True, 5, 256), ((40, 64), 2, 3, True, 0, 64),
            ((33, 24), 3, 9, False, 0, 128), ((17, 16), 4, 1, True, 1, 256), ((8, 8), 33, 5, True, 3, 64)):
        out = []
        for split in (False, True):
            print(f"[paths] mode {mode} channels {channels} {size} spp {spp} frames {frames} "
                  f"split {split}", flush=True)
            r = renderer(capi, vols, tfs, mode, size, spp, 0 if split else 1)
            r.set_frame(size[0], size[1], spp, accumulate, (0.1, 0.2, 0.3))
            r.set_block(block)
            r.set_moments(True)
            if shaded:
                r.set_light((0.3, -1.0, 0.2), True, True)
            if aov:
                r.set_aov(True)
                r.set_aov_frames(aov)
            for _ in range(2):  # the second accumulation runs in cost order
                r.reset_accumulation()
                for _ in range(frames if split else 1):
                    r.render(1 if split else frames)
            got = list(r.read_accum(with_m2=True)) + ([r.read_aov()] if aov else [])
            out.append([g.view(np.uint32) for g in got] + [np.array(list(r.info().values())[3:])])
            r.close()
        for a, b in zip(*out):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("channels,dtype", [(2, np.uint8), (3, np.uint16), (5, np.float16), (9, np.float32)])
@pytest.mark.parametrize("mode", [3, 4, 5, 6, 7, 8])
def test_channels_side_by_side_match_the_oracle(capi, mode, channels, dtype):
    """The modes that read every channel at a position, with channel counts
    that fill their groups of four in part, against the CPU oracle."""
    from oracle import pyoracle
    vols, tfs = volume(channels, dtype, dims=(19, 22, 17))
    print(f"[paths] mode {mode} channels {channels} {np.dtype(dtype)}", flush=True)
    g = renderer(capi, vols, tfs, mode, (43, 30), 1, 1, mc=(4, 5, 3), opacity=0.2)
    o = pyoracle.OracleRenderer()
    for v in vols:
        o.push_channel(v)
    o.init(mode, (4, 5, 3), False)
    for c, t in enumerate(tfs):
        o.set_tf(c, t, 0.2, (0.0, 1.0))
    o.set_frame(43, 30, 1, True, (0.1, 0.2, 0.3))
    o.set_camera(*scenes.orbit_camera(1.6))
    o.set_seed(11)
    g.render(2)
    o.render(2, threads=4)
    np.testing.assert_array_equal(g.read_accum().view(np.uint32), o.read_accum().view(np.uint32))
    g.close()


@pytest.mark.parametrize("conservative", [False, True])
@pytest.mark.parametrize("mode", [1, 3])
@pytest.mark.parametrize("texels", [1, 2, 16, 17, 300])
def test_majorants_match_the_oracle(capi, texels, mode, conservative):
    """Tables shorter and longer than the lanes that share a cell, reversed and
    offset ranges, against the CPU oracle."""
    from oracle import pyoracle
    vols, _ = volume(3, np.uint16, dims=(19, 22, 17))
    rng = np.random.default_rng(texels)
    tfs = [rng.uniform(0, 1, (texels, 4)).astype(np.float32) for _ in vols]
    out = []
    for r in (capi.MdwtRenderer(0), pyoracle.OracleRenderer()):
        for v in vols:
            r.push_channel(v)
        r.init(mode, (9, 7, 8), False)
        r.set_conservative_majorants(conservative)
        for c, (t, xr) in enumerate(zip(tfs, ((0.0, 1.0), (0.8, 0.2), (-0.3, 0.6)))):
            r.set_tf(c, t, 0.7, xr)
        out.append(r.read_majorants().view(np.uint32))
        r.close()
    np.testing.assert_array_equal(out[0], out[1])


@pytest.mark.parametrize("mode", [6, 7, 8, 9])
@pytest.mark.parametrize("texels", [1568, 1572, 3404])
def test_marchers_with_tables_up_to_the_lds(capi, mode, texels):
    """Tables of three channels: the longest with which two workgroups of the
    several-frame kernel fit a CU, the next, and the longest of the one-frame
    kernels (160 KiB with the channel parameters), which the fold's LDS does not
    fit beside."""
    vols, _ = volume(3, np.uint8, dims=(19, 22, 17))
    rng = np.random.default_rng(texels)
    tfs = [rng.uniform(0, 1, (texels, 4)).astype(np.float32) for _ in vols]
    out = []
    for split in (False, True):
        print(f"[paths] mode {mode} texels {texels} split {split}", flush=True)
        r = renderer(capi, vols, tfs, mode, (43, 30), 1, 1, mc=(4, 5, 3), opacity=0.2)
        for _ in range(8 if split else 1):
            r.render(1 if split else 8)
        out.append(r.read_accum().view(np.uint32))
        r.close()
    np.testing.assert_array_equal(*out)


@pytest.mark.parametrize("size,block", [
    ((8, 8), 64), ((16, 8), 128), ((512, 512), 64), ((520, 512), 64), ((1024, 512), 128),
    ((1024, 528), 128), ((1024, 1024), 256), ((1040, 1024), 256)])
def test_cost_order_is_a_permutation(capi, size, block):
    """Frames of one block up to just past 4096, of 64, 128 and 256 pixels: in
    cost order every block is still rendered once (the images of Hilbert order)."""
    vols, tfs = volume(2, np.uint8, dims=(19, 22, 17))
    out = []
    for order in (1, 2):
        print(f"[paths] tile order {order} {size} block {block}", flush=True)
        r = renderer(capi, vols, tfs, 2, size, 1, 1, mc=(4, 5, 3))
        r.set_block(block)
        r.set_tile_order(order)
        images = []
        for _ in range(4):
            r.reset_accumulation()
            r.render(1)
            images.append(r.read_accum().view(np.uint32))
        r.close()
        out.append(images)
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
