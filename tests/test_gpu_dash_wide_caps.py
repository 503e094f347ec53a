"""Round caps of wide dashed strokes, whose arcs have more vertices than a wavefront keeps at a time: on the GPU
against the oracle on both sides of that limit (a half circle of 128 vertices is one of half-width 320), with
pieces of one and of several rounds of 64 caps, starting and ending in dashes and gaps; and their geometry
takes time in proportion to the vertices."""
import math

import numpy as np
import pytest

from vkvg_amd import scenes
from vkvg_amd.stream import CAP_ROUND, Stream

pytestmark = pytest.mark.gpu


def _line(s, caps, hw, dashes, offset, angle, through):
    """A dashed line of about that many caps that ends half a width before the point, so that the arcs of its
    last caps cross the surface, and a short segment after it."""
    length = caps * sum(dashes) / len(dashes)
    d = np.array([math.cos(angle), math.sin(angle)])
    end = np.asarray(through) - hw * d
    s.set_line_width(2 * hw)
    s.set_line_cap(CAP_ROUND)
    s.set_dash(dashes, offset)
    s.polyline(np.array([end - length * d, end, end + [9.5, 4.25]], np.float32))
    s.stroke()


@pytest.mark.parametrize("hw,counts", [(318.0, (5, 70)), (320.0, (5, 70)), (322.5, (5, 70)), (1000.0, (4, 64, 131)),
                                       (4000.0, (5, 66)), (16000.0, (6, 65))])
def test_wide_round_caps_equal_the_oracle(hw, counts):
    import vkvg_amd
    from parity_util import compare, render_gpu, render_oracle
    size = 160
    rng = scenes.Rng(int(hw))
    s = Stream()
    s.set_source_rgb(1, 1, 1)
    s.paint()
    for i, n in enumerate(counts):
        s.set_source_rgba(*rng.u(3), 0.02)
        _line(s, n, hw, [7.0, 4.5], float(rng.uniform(0, 11)), float(rng.uniform(0, 6.28)), rng.uniform(40, 120, 2))
    sc = scenes.Scene("wide_caps", size, size, s, len(counts))
    rgba, sig, _ = render_oracle(sc)
    assert len(np.unique(sig)) > 8  # outlines of several caps cross the surface
    with vkvg_amd.Device() as dev:
        g_rgba, g_sig, _ = render_gpu(dev, sc)
    r = compare(g_rgba, g_sig, rgba, sig)
    assert r["mask_mismatch_px"] == 0 and r["rgba_max_err"] == 0, r


def test_cost_of_wide_round_caps_is_linear_in_their_vertices(device):
    """Half-widths of 4000 and 16000 px (1600 and 6400 vertices per half circle): at most four times the time, and
    what does not grow makes it less. Work per vertex that grows with the vertex's place gives 16."""
    import vkvg_amd
    ms = {}
    for hw in (4000.0, 16000.0):
        s = Stream()
        s.set_source_rgba(0, 0, 0, 0.5)
        _line(s, 66, hw, [7.0, 4.5], 3.0, 0.7, (-50000.0, -50000.0))  # off the surface: geometry alone
        surf = vkvg_amd.Surface(device, 64, 64)
        surf.upload(s.words())
        t = []
        for _ in range(6):
            vkvg_amd.execute(device)
            t.append(device.stats()["ms_stage"]["geometry"])
        surf.close()
        ms[hw] = min(t)
    print(ms, flush=True)
    assert ms[16000.0] < 8 * ms[4000.0], ms
