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
