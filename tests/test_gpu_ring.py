"""Copies through the pinned ring that are longer than the ring, both ways,
against data that took another way; and the ring beside a thread's older errors."""
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


def _rgba8(accum):
    v = np.clip(np.trunc(np.clip(accum * np.float32(256), -1, 256)), 0, 255).astype(np.uint32)
    return v[..., 0] | (v[..., 1] << 8) | (v[..., 2] << 16) | (v[..., 3] << 24)


# float images of 16 MiB and 32 KiB, and of 34.3 MiB (the ring's 16 MiB twice and
# a tail). Their 8-bit images are a quarter of that, so a float pixel that lies in
# a slot's second chunk has its 8-bit one in a first.
@pytest.mark.parametrize("w,h", [(1026, 1024), (1500, 1501)])
def test_images_longer_than_the_ring(capi, w, h):
    print(f"[ring] {w} x {h}", flush=True)
    r = _renderer(capi, w, h)
    r.render(1)
    a, m2 = r.read_accum(with_m2=True)
    assert len(np.unique(a[..., 0])) > 1
    np.testing.assert_array_equal(_rgba8(a), r.read_fb())
    np.testing.assert_array_equal(m2, a * a)
    r.close()


def test_channel_longer_than_the_ring(capi):
    """A channel of 42.3 MB (two and a half rings, an odd tail) of random bytes:
    the value ranges of its cells against the oracle's."""
    from oracle import pyoracle
    vol = np.random.default_rng(5).integers(0, 256, (349, 347, 349), dtype=np.uint8)
    vol[::2] //= 2  # ranges that differ between cells of one layer too
    vol[:, 1::3] //= 3
    out = []
    for r in (capi.MdwtRenderer(0), pyoracle.OracleRenderer()):
        r.push_channel(vol)
        r.init(2, (117, 119, 116), False)
        out.append(r.read_ranges())
        r.close()
    assert len(np.unique(out[1])) > 50
    np.testing.assert_array_equal(*out)


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
