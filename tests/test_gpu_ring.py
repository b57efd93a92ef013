"""Copies through the pinned ring beside a thread's older errors."""
import ctypes

import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    from mdwtracker_amd import capi
    return capi


def _renderer(capi, w, h):
    r = capi.MdwtRenderer(0)
    rng = np.random.default_rng(3)
    r.push_channel(scenes.blob_volume_u8(24, 5, rng))
    r.init(2, (4, 4, 4), True)
    r.set_tf(0, scenes.piecewise_tf(4, rng, 0.3, clear_first=True), 0.2, (0.0, 1.0))
    r.set_frame(w, h, 1, True, (0.2, 0.4, 0.6))
    r.set_moments(True)
    return r


def test_after_an_error_of_the_thread(capi):
    """An error that another use of the runtime left on the thread is not the
    copy's."""
    r = _renderer(capi, 725, 727)
    r.render(1)
    want = r.read_accum()
    hip = ctypes.CDLL("libamdhip64.so.7")  # the library that libmdwt.so has loaded
    assert hip.hipSetDevice(9999) != 0  # refused by the runtime, which keeps the error
    np.testing.assert_array_equal(r.read_accum(), want)
    hip.hipGetLastError()
    r.close()
