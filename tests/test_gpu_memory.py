"""Device memory that is short: what a handle keeps for speed alone makes room.
Most of the card is taken by one allocation of the test's own, freed after it."""
import ctypes
import gc
from contextlib import contextmanager

import numpy as np
import pytest

from mdwtracker_amd import scenes

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.fixture(scope="module")
def capi():
    from mdwtracker_amd import capi
    return capi


@pytest.fixture(scope="module")
def hip(capi):
    return ctypes.CDLL("libamdhip64.so.7")  # the runtime that libmdwt.so has loaded


def _memory(hip):
    """(free, total) bytes of the device"""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value, total.value


def _take(hip, left):
    """Allocations that leave `left` bytes of the device free (in a few steps: the
    runtime counts more as free at first than it has)."""
    taken = []
    for _ in range(4):
        n = _memory(hip)[0] - left
        if n < 8 * MIB:
            break
        p = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(n)) == 0
        taken.append(p)
    return taken


@pytest.fixture(scope="module", autouse=True)
def most_of_the_card(hip):
    taken = _take(hip, 48 << 30)
    yield
    for p in taken:
        assert hip.hipFree(p) == 0


def _alloc(hip, n):
    p = ctypes.c_void_p()
    if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(n)) == 0:
        return p
    hip.hipGetLastError()
    return None


@contextmanager
def _only(hip, left):
    gc.collect()  # handles that other tests left to the collector
    taken = _take(hip, left)
    # memory that the runtime can still give beside what it counts as free
    hidden = 0
    while hidden < 8 << 30:
        p = _alloc(hip, left + hidden + 64 * MIB)
        if p is None:
            break
        assert hip.hipFree(p) == 0
        hidden += 64 * MIB
    if hidden:
        taken.append(_alloc(hip, hidden))
        assert taken[-1] is not None
    try:
        print(f"[memory] free {_memory(hip)[0] >> 20} MiB, hidden {hidden >> 20} MiB", flush=True)
        assert abs(_memory(hip)[0] - left) < 16 * MIB or hidden
        yield
    finally:
        for p in taken:
            assert hip.hipFree(p) == 0


def _renderer(capi, mode, dims=(64, 48, 40), size=(96, 64)):
    """Two u8 channels of `dims` voxels: their joint copy has 4 bytes a voxel."""
    rng = np.random.default_rng(9)
    r = capi.MdwtRenderer(0)
    for _ in range(2):
        block = scenes.blob_volume_u8(16, 5, rng)
        reps = [-(-n // 16) for n in dims[::-1]]
        r.push_channel(np.ascontiguousarray(np.tile(block, reps)[:dims[2], :dims[1], :dims[0]]))
    r.init(mode, (8, 8, 8), True)
    for c in range(2):
        r.set_tf(c, scenes.piecewise_tf(6, rng, 0.3 * c, clear_first=True), 0.2, (0.0, 1.0))
    r.set_frame(size[0], size[1], 1, True, (0.2, 0.4, 0.6))
    r.set_seed(5)
    r.render(1)  # what the runtime allocates at a first launch is there
    r.reset_accumulation()
    return r


def test_frame_without_room_for_its_8_bit_image(capi, hip):
    """A frame whose accumulator fits beside nothing else: rendered and read as
    floats; the 8-bit image is refused, and read once there is memory."""
    r = _renderer(capi, 2)
    with _only(hip, 1024 * MIB + 128 * MIB):
        r.set_frame(8192, 8192, 1, True, (0.2, 0.4, 0.6))  # 1 GiB, and 256 MiB as RGBA8
        r.render(1)
        a = r.read_accum()
        with pytest.raises(Exception, match="RGBA8"):
            r.read_fb()
    v = np.clip(np.trunc(np.clip(a * np.float32(256), -1, 256)), 0, 255).astype(np.uint32)
    np.testing.assert_array_equal(v[..., 0] | (v[..., 1] << 8) | (v[..., 2] << 16) | (v[..., 3] << 24), r.read_fb())
    r.close()


def test_a_frame_that_was_not_allocated_is_an_error(capi, hip):
    """A frame that does not fit is refused, and so is rendering until one does."""
    r = _renderer(capi, 2)
    r.render(1)
    want = r.read_accum()
    with _only(hip, 512 * MIB):
        with pytest.raises(Exception):
            r.set_frame(8192, 8192, 1, True, (0.2, 0.4, 0.6))
        for _ in range(2):
            with pytest.raises(Exception):
                r.render(1)
    r.set_frame(96, 64, 1, True, (0.2, 0.4, 0.6))
    r.render(1)
    assert r.read_accum().shape == want.shape
    r.close()


def test_joint_copy_goes_with_the_modes_that_read_it(capi, hip):
    dims = (512, 512, 256)
    joint = 4 * dims[0] * dims[1] * dims[2]  # 256 MiB
    r = _renderer(capi, 2, dims)
    base = _memory(hip)[0]
    for mode, has in ((3, True), (8, True), (9, False), (4, True), (1, False)):
        r.set_mode(mode)
        assert abs(base - _memory(hip)[0] - has * joint) < 16 * MIB, mode
    r.close()


@pytest.mark.parametrize("mode", [3, 5, 7])
def test_joint_copy_leaves_a_reserve(capi, hip, mode):
    """Not made where less than an eighth of the device would be left; the same
    images from the channels' own bricks."""
    dims = (512, 512, 256)
    r = _renderer(capi, 2, dims)
    r.set_mode(mode)
    r.render(3)
    want = r.read_accum()
    r.close()
    r = _renderer(capi, 2, dims)
    with _only(hip, _memory(hip)[1] // 8 + 128 * MIB):
        base = _memory(hip)[0]
        r.set_mode(mode)
        assert abs(base - _memory(hip)[0]) < 16 * MIB
        r.render(3)
        got = r.read_accum()
    assert want[..., :3].std() > 0.01
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    r.close()


@pytest.mark.parametrize("views", [False, True])
def test_joint_copy_makes_room(capi, hip, views):
    """A frame, or views, that fit only where the joint copy was (1.5 GiB), with the
    images of a handle that has both; a graph captured with it is not replayed."""
    dims = (1024, 768, 512)
    joint = 4 * dims[0] * dims[1] * dims[2]
    view = {"from": (0.5, 0.6, 2.4), "at": (0.5, 0.5, 0.5), "up": (0.0, 1.0, 0.0), "fovy": 45.0, "width": 8192,
            "height": 8192, "spp": 1, "seed": 3}
    small = dict(view, width=96, height=64)
    out = []
    for short in (False, True):
        r = _renderer(capi, 3, dims)
        r.batch_set_launch(2)
        r.batch_set_views([small])
        r.batch_render(2)  # captures the graph
        base = _memory(hip)[0]
        if short:
            with _only(hip, 640 * MIB):
                if views:
                    r.batch_set_views([small, view])
                else:
                    r.set_frame(8192, 8192, 1, True, (0.2, 0.4, 0.6))
                # the copy went, 1 GiB of accumulators came (and up to 256 MiB of RGBA8)
                assert _memory(hip)[0] > 640 * MIB + joint - 1024 * MIB - 300 * MIB
                r.batch_render(2)
                if not views:
                    r.render(1)
        else:
            if views:
                r.batch_set_views([small, view])
            else:
                r.set_frame(8192, 8192, 1, True, (0.2, 0.4, 0.6))
            assert base - _memory(hip)[0] > 1024 * MIB
            r.batch_render(2)
            if not views:
                r.render(1)
        out.append([r.batch_read_view(0)] + [r.batch_read_view(1) if views else r.read_accum()])
        r.close()
    for a, b in zip(*out):
        assert a[..., :3].std() > 0.01
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
