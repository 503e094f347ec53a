"""Dashed pieces emitted by one thread or by a wavefront, on the GPU against the oracle: cap counts around
the thresholds and around the 64 caps of a wavefront's round, every cap style, closed and open sub-paths
(final caps, joins at pieces that start in a gap), arcs of more vertices than a wavefront keeps, dash
arrays of 1, 2, 5 and 70 entries, and frames of few and of many stroke steps."""
import math

import numpy as np
import pytest

from vkvg_amd.stream import Stream
from vkvg_amd import scenes

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 3, 4, 5, 14, 15, 16, 17, 31, 33, 62, 63, 64, 65, 66, 127, 128, 129, 200]


def _scene(cap, dashes, many, width=6.0, size=900):
    rng = scenes.Rng(77 + cap)
    s = Stream()
    s.set_source_rgb(1, 1, 1)
    s.paint()
    if many:  # solid steps beyond the line between few and many
        xy = np.stack([rng.uniform(0, size, 17000), rng.uniform(0, 4, 17000)], 1)
        s.set_line_width(0.5)
        s.set_source_rgba(0, 0, 0, 0.01)
        s.polyline(xy)
        s.stroke()
    s.set_line_cap(cap)
    s.set_line_width(width)
    mean = float(sum(dashes)) / len(dashes)
    for i, n in enumerate(COUNTS):
        s.set_line_join(i % 3)
        s.set_dash(dashes, float(rng.uniform(0, 2 * mean)))
        s.set_source_rgba(*rng.u(3), float(rng.uniform(0.4, 1)))
        a, length = float(rng.uniform(0, 2 * math.pi)), n * mean
        x, y = float(rng.uniform(0, size)), float(rng.uniform(0, size))
        p = [(x, y), (x + length * math.cos(a), y + length * math.sin(a))]
        a += float(rng.uniform(0.5, 2.5))
        p.append((p[1][0] + 0.7 * length * math.cos(a), p[1][1] + 0.7 * length * math.sin(a)))
        s.polyline(np.array(p, np.float32), close=i % 2 == 1)
        s.stroke()
    return scenes.Scene("dash_pieces", size, size, s, len(COUNTS))


@pytest.mark.parametrize("many", [False, True], ids=["few", "many"])
@pytest.mark.parametrize("cap", [0, 1, 2], ids=["butt", "round", "square"])
@pytest.mark.parametrize("dashes", [[7.0], [8.0, 4.0], [3.3, 1.7, 0.0, 2.9, 5.1]], ids=["1", "2", "5"])
def test_piece_sizes(cap, dashes, many):
    _check(_scene(cap, dashes, many))


def test_wide_round_caps_and_long_dash_array():
    _check(_scene(1, [40.0, 25.0], False, width=1500.0))  # arcs beyond the kept vertices
    _check(_scene(1, [2.0 + 0.13 * i for i in range(70)], False))  # more dashes than lanes


def _check(sc):
    import vkvg_amd
    from parity_util import compare, render_gpu, render_oracle
    rgba, sig, _ = render_oracle(sc)
    with vkvg_amd.Device() as dev:
        g_rgba, g_sig, _ = render_gpu(dev, sc)
    r = compare(g_rgba, g_sig, rgba, sig)
    assert r["mask_mismatch_px"] == 0 and r["rgba_max_err"] == 0, r
