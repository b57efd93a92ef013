"""Batched views of one handle whose mode, lighting and schedule change between
frames, in every launch form, against a handle of its own for each."""
import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from mdwtracker_amd import capi
    return capi


VIEWS = [{"from": (0.5 + 1.8 * np.sin(a), 0.7, 0.5 + 1.8 * np.cos(a)), "at": (0.5, 0.5, 0.5), "up": (0.0, 1.0, 0.0),
          "fovy": 45.0, "width": w, "height": h, "spp": s, "seed": 7 + w}
         for a, w, h, s in ((0.3, 57, 40, 1), (2.1, 33, 64, 2))]


def _handle(capi, launch):
    r = capi.MdwtRenderer(0)
    rng = np.random.default_rng(4)
    for _ in range(2):
        r.push_channel(scenes.blob_volume_u8(24, 5, rng))
    r.init(2, (4, 4, 4), True)
    for c in range(2):
        r.set_tf(c, scenes.piecewise_tf(6, rng, 0.4 * c, clear_first=True), 0.3, (0.0, 1.0))
    r.batch_set_launch(launch)
    r.batch_set_views(VIEWS)
    return r


def _frames(r, mode, lit, schedule):
    r.set_mode(mode)
    r.set_light((0.3, -1.0, 0.2), lit, lit)
    r.set_schedule(schedule)
    r.batch_reset()
    r.batch_render(2)
    return [r.batch_read_view(i) for i in range(len(VIEWS))]


@pytest.mark.parametrize("launch", [0, 1, 2])
@pytest.mark.parametrize("lit", [False, True])
def test_changes_between_batched_frames(capi, launch, lit):
    """The frame ids run on over a reset, so each fresh handle first renders as many
    frames as the changing one has."""
    r = _handle(capi, launch)
    steps = [(m, s) for m in (2, 0, 1, 3, 5, 4, 8, 6, 9, 7) for s in (1, 0)]
    before = 0
    for mode, schedule in steps:
        print(f"[batch] launch {launch} lit {lit} mode {mode} schedule {schedule}", flush=True)
        got = _frames(r, mode, lit, schedule)
        f = _handle(capi, launch)
        if before:
            f.batch_render(before)
        want = _frames(f, mode, lit, schedule)
        f.close()
        before += 2
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
    r.close()
