"""Images and network inputs copied through the pinned ring: sizes around its
chunks and pieces, and several threads with handles of their own."""
import threading

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


def _fb_of(accum):
    """make_rgba of the float image (the reference's 8-bit conversion)"""
    v = np.clip(np.trunc(np.clip(accum * np.float32(256), -1, 256)), 0, 255).astype(np.uint32)
    return v[..., 0] | (v[..., 1] << 8) | (v[..., 2] << 16) | (v[..., 3] << 24)


def _fb_noalloc(capi, r):
    out = np.empty((r.height, r.width), np.uint32)
    assert capi.lib.mdwt_read_fb_noalloc(r._h, out.ctypes.data_as(capi._up)) == 0
    return out


# bytes of the 8-bit / float image: below one piece, one byte-sized tail past
# 512 KiB, one chunk, a chunk and a tail, more chunks than the ring has slots
@pytest.mark.parametrize("w,h", [(3, 5), (367, 359), (512, 1024), (725, 727), (1021, 1019)])
def test_read_back_sizes(capi, w, h):
    print(f"[copy] {w} x {h}", flush=True)
    r = _renderer(capi, w, h)
    for _ in range(2):
        r.render(1)
        a, m2 = r.read_accum(with_m2=True)
        want = _fb_noalloc(capi, r)
        np.testing.assert_array_equal(_fb_of(a), want)
        np.testing.assert_array_equal(r.read_fb(), want)
        if r.info()["accum_id"] == 1:  # one frame: the second moment is the square
            np.testing.assert_array_equal(m2, a * a)
    r.close()


def test_threads_with_handles_of_their_own(capi):
    """More threads than lanes, reading and denoising side by side."""
    from mdwtracker_amd import denoise
    errors = []

    def work(k):
        try:
            r = _renderer(capi, 640 + 8 * k, 700)
            dn = denoise.Denoiser(320, 256, seed=2)
            x = np.random.default_rng(7).random((256, 320, 11), np.float32)
            first = dn.infer(x)[0]
            for _ in range(6):
                r.render(1)
                np.testing.assert_array_equal(_fb_of(r.read_accum()), r.read_fb())
                np.testing.assert_array_equal(dn.infer(x)[0], first)
            r.close()
            dn.close()
        except Exception as e:  # reported by the main thread
            errors.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
