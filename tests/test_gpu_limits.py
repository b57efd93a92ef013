"""Calls at the limits of their arguments."""
import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from mdwtracker_amd import capi
    return capi


def _renderer(capi, mode=2, channels=1, dim=24):
    r = capi.MdwtRenderer(0)
    rng = np.random.default_rng(3)
    for _ in range(channels):
        r.push_channel(scenes.blob_volume_u8(dim, 5, rng))
    r.init(mode, (4, 4, 4), True)
    for c in range(channels):
        r.set_tf(c, scenes.piecewise_tf(4, rng, 0.3, clear_first=True), 0.2, (0.0, 1.0))
    r.set_seed(17)
    return r


def test_frame_of_2_30_pixels(capi):
    """The largest frame: four frames in one call, whose several-frame launch
    would have 2^32 threads, against four calls."""
    out = []
    for split in (False, True):
        print(f"[limits] 32768 x 32768 split {split}", flush=True)
        r = _renderer(capi)
        r.set_frame(32768, 32768, 1, True, (0.2, 0.4, 0.6))
        for _ in range(4 if split else 1):
            r.render(1 if split else 4)
        out.append(r.read_fb())
        r.close()
    assert len(np.unique(out[0][16384, ::64])) > 1  # the volume is hit: up to five levels in four frames
    assert np.array_equal(*out)


@pytest.mark.parametrize("launch", [0, 1])
def test_batch_of_2_30_pixels(capi, launch):
    """4096 views of 512^2, four frames in one call, against single-view renders."""
    views = []
    for i in range(4096):
        th = 2 * np.pi * i / 4096
        views.append({"from": (0.5 + 2.2 * np.sin(th), 0.7, 0.5 + 2.2 * np.cos(th)), "at": (0.5, 0.5, 0.5),
                      "up": (0.0, 1.0, 0.0), "fovy": 40.0, "width": 512, "height": 512, "spp": 1, "seed": i})
    print(f"[limits] 4096 views launch {launch}", flush=True)
    g = _renderer(capi)
    g.batch_set_launch(launch)
    g.batch_set_views(views)
    g.batch_render(4)
    for i in (0, 1365, 4095):
        v = views[i]
        s = _renderer(capi)
        s.set_frame(512, 512, 1, True, (0.0, 0.0, 0.0))
        s.set_camera(v["from"], v["at"], v["up"], v["fovy"])
        s.set_seed(v["seed"])
        s.render(4)
        want = s.read_accum()
        s.close()
        assert want[..., :3].std() > 0.01
        np.testing.assert_array_equal(g.batch_read_view(i).view(np.uint32), want.view(np.uint32))
    g.close()


@pytest.mark.parametrize("channels,size", [(1, (2365, 2365)), (5, (1549, 1547)), (12, (1095, 1095)), (12, (1094, 1095))])
def test_auxiliary_buffers_of_more_than_a_piece(capi, channels, size):
    """Around the 64 MiB piece of the packed read-back, with the buffers' rows
    padded: a pixel misses exactly where the image shows the background."""
    print(f"[limits] aov {channels} channels {size}", flush=True)
    bg = (0.3137, 0.41, 0.77)
    r = _renderer(capi, mode=2, channels=channels)
    r.set_aov(True)
    r.set_frame(size[0], size[1], 1, True, bg)
    r.set_camera((0.5, 0.5, 0.05), (0.5, 0.5, 1.0), (0.0, 1.0, 0.0), 60.0)  # inside: every ray is in the volume
    r.render(1)
    img, aov = r.read_accum(), r.read_aov()
    r.close()
    miss = (img[..., :3] == np.float32(bg)).all(-1)
    assert 0.0 < miss.mean() < 1.0 and not miss[-1].all()
    np.testing.assert_array_equal(aov[..., 1], miss.astype(np.float32))
    np.testing.assert_array_equal(aov[..., 1:].sum(-1), np.ones(miss.shape, np.float32))
    # the first free flight may have no length: a hit at 0, with odds of about 1e-7 a step
    assert (aov[..., 0][miss] == 0).all() and (aov[..., 0][~miss] > 0).mean() > 0.9999
