"""Flattening on the GPU against the oracle on both sides of the limit up to which a frame's cubics are
split over several threads (65536, with 64 points per part up to 16384 and 32 beyond), with cubics of a
few to several thousand points (parts that overflow), and lines and arcs among them."""
import numpy as np
import pytest

from vkvg_amd import scenes
from vkvg_amd.stream import Stream

pytestmark = pytest.mark.gpu


def _scene(n_small, big, size=320):
    """n_small tiny cubics in closed paths of up to 100, then `big` cubics up to 20 000 px long."""
    rng = scenes.Rng(5 + n_small)
    s = Stream()
    s.set_source_rgb(1, 1, 1)
    s.paint()
    left = n_small
    while left:
        n = min(left, 100)
        c = rng.uniform(0, size, 2)
        pts = (np.tile(c, 1 + 3 * n) + rng.uniform(-12, 12, 2 + 6 * n)).astype(np.float32)
        s.set_source_rgba(*rng.u(3), 0.3)
        s.curves(pts[:2], pts[2:].reshape(n, 6), close=True)
        s.fill()
        left -= n
    s.set_line_width(2.0)
    for k in range(big):
        r = 10.0 ** (1.5 + 2.8 * k / max(1, big - 1))
        p = (size / 2 + r * (2 * rng.u(8) - 1)).astype(np.float32)
        s.set_source_rgba(*rng.u(3), 0.5)
        s.move_to(float(p[0]), float(p[1]))
        s.curve_to(*[float(v) for v in p[2:]])
        s.line_to(float(p[0]) + 9, float(p[3]))
        s.arc(float(size / 2), float(size / 2), 5.0 + k, 0.0, 4.0)
        s.stroke()
    return scenes.Scene("flatten_split", size, size, s, 1)


@pytest.mark.parametrize("n_small,big", [(0, 0), (0, 1), (7, 0), (8, 12), (9, 30), (16384 - 12, 12), (16385, 0),
                                         (65536 - 12, 12), (65537, 0)])
def test_frames_of_few_and_many_cubics(n_small, big):
    import vkvg_amd
    from parity_util import compare, render_gpu, render_oracle
    sc = _scene(n_small, big)
    rgba, sig, _ = render_oracle(sc)
    with vkvg_amd.Device() as dev:
        g_rgba, g_sig, _ = render_gpu(dev, sc)
    r = compare(g_rgba, g_sig, rgba, sig)
    assert r["mask_mismatch_px"] == 0 and r["rgba_max_err"] == 0, r
