"""Frames that outgrow the buffers of the frames before them on the same engine, in path tiles, segments,
commands or all of them, and frames after them that do not: the pass that counts them runs with the buffers as
they are, leaves out what does not fit and runs again."""
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
