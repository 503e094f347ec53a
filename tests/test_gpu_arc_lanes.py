"""Arcs shared out over a wavefront's lanes, against the oracle: frames whose wavefronts hold one, a few,
eight, nine and 64 and more arcs, of fewer, as many and more points than lanes, circles and ellipses,
with lines and cubics among them."""
import math

import pytest

from vkvg_amd import scenes
from vkvg_amd.stream import Stream

pytestmark = pytest.mark.gpu


def _scene(arcs, rmax, between, size=300):
    rng = scenes.Rng(900 + arcs + between)
    s = Stream()
    s.set_source_rgb(1, 1, 1)
    s.paint()
    s.set_line_width(1.5)
    for k in range(arcs):
        r = rmax * (k + 1) / arcs
        x, y, a = float(rng.uniform(0, size)), float(rng.uniform(0, size)), float(rng.uniform(-7, 7))
        s.set_source_rgba(*rng.u(3), 0.4)
        s.move_to(x, y)
        for j in range(between):
            s.line_to(x + 3 * j, y + 5 * (j % 3))
        if k % 5 == 4:
            s.elliptic_arc_to(x + r, y + r / 3, bool(k % 2), bool(k % 3), 0.8 * r, 0.4 * r, a)
        elif k % 5 == 3:
            s.arc_negative(x, y, r, a, a - 2 * math.pi)
        elif k % 5 == 2:
            s.curve_to(x + r, y, x, y + r, x + 9, y + 9)
            s.arc(x, y, r, a, a + 0.3)
        else:
            s.arc(x, y, r, a, a + 2 * math.pi)
        s.fill_preserve() if k % 2 else s.stroke()
        s.new_path()
    return scenes.Scene("arc_lanes", size, size, s, 1)


@pytest.mark.parametrize("arcs,rmax,between", [(1, 400.0, 0), (1, 1.0, 80), (2, 4000.0, 0), (7, 90.0, 9), (8, 30.0, 3),
                                               (9, 300.0, 3), (63, 40.0, 0), (65, 700.0, 0), (200, 12.0, 1)])
def test_arcs_over_lanes(arcs, rmax, between):
    import vkvg_amd
    from parity_util import compare, render_gpu, render_oracle
    sc = _scene(arcs, rmax, between)
    rgba, sig, _ = render_oracle(sc)
    with vkvg_amd.Device() as dev:
        g_rgba, g_sig, _ = render_gpu(dev, sc)
    r = compare(g_rgba, g_sig, rgba, sig)
    assert r["mask_mismatch_px"] == 0 and r["rgba_max_err"] == 0, r
