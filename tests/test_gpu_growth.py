"""Frames that outgrow the buffers of the frames before them on the same engine, in path tiles, segments,
commands or all of them, and frames after them that do not: the pass that counts them runs with the buffers as
they are, counts what does not fit without writing it, and is followed by one more that writes everything."""
import ctypes

import numpy as np
import pytest

from vkvg_amd import scenes
from vkvg_amd.stream import Stream

pytestmark = pytest.mark.gpu


def _scene(n, size, extent, clip=False):
    """n filled triangles of up to `extent` pixels on a painted ground: path tiles by extent, segments by n."""
    rng = scenes.Rng(31 + n + size)
    s = Stream()
    s.set_source_rgb(0.9, 0.9, 0.8)
    s.paint()
    if clip:
        s.rectangle(3, 5, size * 0.8, size * 0.9)
        s.clip()
    for _ in range(n):
        c = rng.uniform(0, size, 2)
        p = c + rng.uniform(-extent, extent, 6).reshape(3, 2)
        s.set_source_rgba(*rng.u(3), 0.4)
        s.move_to(float(p[0][0]), float(p[0][1]))
        s.line_to(float(p[1][0]), float(p[1][1]))
        s.line_to(float(p[2][0]), float(p[2][1]))
        s.fill()
    return scenes.Scene("growth", size, size, s, 1)


def test_frames_outgrow_their_buffers():
    import vkvg_amd
    from parity_util import compare, render_gpu, render_oracle
    with vkvg_amd.Device() as dev:
        for n, size, extent, clip in ((1, 40, 9, False), (3, 400, 300, False), (4000, 90, 5, False), (600, 700, 60, True),
                                      (2, 30, 6, True), (900, 1000, 500, False), (0, 64, 1, False)):
            sc = _scene(n, size, extent, clip)
            rgba, sig, _ = render_oracle(sc)
            g_rgba, g_sig, _ = render_gpu(dev, sc)
            r = compare(g_rgba, g_sig, rgba, sig)
            assert r["mask_mismatch_px"] == 0 and r["rgba_max_err"] == 0, (n, size, extent, r)


@pytest.mark.parametrize("size,n", [(1440, 3), (1456, 3), (200, 8191), (200, 8192), (200, 8193)])
def test_work_order_of_one_workgroup_and_of_many(size, n):
    """8100 and 8281 tiles, and 8192 to 8194 draws with the paint: both sides of the limit of 8192"""
    import vkvg_amd
    from parity_util import compare, render_gpu, render_oracle
    sc = _scene(n, size, 200 if size > 1000 else 4)
    rgba, sig, _ = render_oracle(sc)
    with vkvg_amd.Device() as dev:
        g_rgba, g_sig, _ = render_gpu(dev, sc)
    r = compare(g_rgba, g_sig, rgba, sig)
    assert r["mask_mismatch_px"] == 0 and r["rgba_max_err"] == 0, r


def test_outgrown_buffers_cost_one_more_binning_and_no_wait():
    """Three waits for counts in every frame; the draws of a frame that outgrows path tiles, segments or both are
    binned twice, those of one that outgrows nothing once."""
    import vkvg_amd
    L = vkvg_amd.lib()
    passes = L.vkh_last_frame_passes
    passes.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_uint32)]
    passes.restype = None
    out = (ctypes.c_uint32 * 2)()
    most = np.array([24, 400])  # path tiles and segments that a new engine's buffers hold, rounded up
    outgrown = set()
    with vkvg_amd.Device() as dev:
        for n, size, extent in [(60, 80, 20), (4000, 200, 9), (40, 2000, 1700), (40000, 200, 6), (30000, 1000, 60)]:
            s = vkvg_amd.Surface(dev, size, size)
            s.upload(_scene(n, size, extent).words())
            for times in (2, 1):  # it outgrows the buffers, and then no more
                vkvg_amd.execute(dev)
                passes(dev._engine(), out)
                assert list(out) == [3, times], (n, size, extent, list(out))
            s.close()
            st = dev.stats()
            counts = np.array([st["path_tiles"], st["segments"]])
            print(n, size, extent, counts, most)
            outgrown.add(tuple(counts > 1.6 * most))  # a buffer grows to half as much again as needed
            most = np.maximum(most, counts)
    assert outgrown >= {(True, False), (False, True), (True, True)}, outgrown


def test_more_path_tiles_than_32_bits_are_refused():
    """1025 slivers across a 32768x32768 surface: 2048x2048 tiles of 16 pixels each, 2^32 + 2^22 path tiles, whose
    32-bit sum would be 2^22. The frame is refused and the next one renders."""
    import vkvg_amd
    s = Stream()
    s.set_source_rgba(0, 0, 0, 1)
    for _ in range(1025):
        s.move_to(0.5, 0.5)
        s.line_to(32767.5, 32767.5)
        s.line_to(32767.5, 32766.5)
        s.fill()
    t = Stream()
    t.set_source_rgba(0, 0, 1, 1)
    t.rectangle(100, 100, 8, 8)
    t.fill()
    with vkvg_amd.Device() as dev:
        surf = vkvg_amd.Surface(dev, 32768, 32768)
        surf.upload(s.words())
        with pytest.raises(vkvg_amd.VkvgError):
            vkvg_amd.execute(dev)
        L = vkvg_amd.lib()
        L.vkvg_hip_last_error.restype = ctypes.c_char_p
        L.vkvg_hip_last_error.argtypes = [ctypes.c_void_p]
        assert b"path tiles" in L.vkvg_hip_last_error(dev._engine())
        small = vkvg_amd.Surface(dev, 128, 128)
        small.replay(t.words())
        assert small.premultiplied()[104, 104].tolist() == [0, 0, 255, 255]
        small.close()
        surf.close()
