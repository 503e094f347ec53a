"""The fine kernel's variants on the GPU against the oracle: tiles of 8, 16 and 32 pixels at every batch
capacity, frames on both sides of the line between the wide and the narrow workgroup of 16-pixel tiles
(4096 tiles), with and without coverage signatures, on surfaces whose sizes leave partial tiles."""
import numpy as np
import pytest

from oracle import ovg
from vkvg_amd import scenes
from vkvg_amd.stream import Stream

pytestmark = pytest.mark.gpu

_REF = {}


def _scene(kind, size):
    if kind == "stack":  # 150 layers over every tile: more than the 64 commands staged at a time
        rng, s = scenes.Rng(9), Stream()
        for i in range(150):
            s.set_operator(3 if i % 11 == 5 else 2)
            if i % 7 == 3:
                s.set_linear(*rng.uniform(0, size, 4), [(0.0, *rng.u(3), 0.1), (0.6, *rng.u(3), 0.2), (1.0, *rng.u(3), 0.1)])
            else:
                s.set_source_rgba(*rng.u(3), 0.1)
            s.set_fill_rule(i % 2)
            s.polyline(rng.uniform(-size / 2, 1.5 * size, 10).reshape(5, 2), close=True)
            if i % 3:
                s.rectangle(-1, -1, size + 2, size + 2)
            if i % 5 == 4:
                s.set_line_width(float(rng.uniform(1, 9)))
                s.stroke()
            else:
                s.fill()
        return scenes.Scene("stack", size, size, s, 150), []
    if kind == "mix":  # every operator, clips, surface sources, even-odd and non-zero fills, strokes
        return scenes.grand_mix(variant=3, size=size, n=80)
    return scenes.config3(variant=2, n_paths=120, size=size), []  # solid and gradient fills and strokes


def _reference(kind, size):
    if (kind, size) not in _REF:
        sc, src = _scene(kind, size)
        _REF[kind, size] = ovg.render(size, size, sc.words(), sources=src)[:2]
    return _REF[kind, size]


@pytest.mark.parametrize("kind", ["mix", "dense", "stack"])
@pytest.mark.parametrize("size", [61, 1023, 1041])  # 1023: 4096 tiles of 16 pixels; 1041: 4356
@pytest.mark.parametrize("tile", [8, 16, 32])
@pytest.mark.parametrize("words", [2048, 4096, 8192])
def test_fine_variants_equal_the_oracle(kind, size, tile, words):
    import vkvg_amd
    rgba, sig = _reference(kind, size)
    sc, bitmaps = _scene(kind, size)
    with vkvg_amd.Device() as dev:
        dev.set_tile_size(tile)
        dev.set_fine_words(words)
        srcs = [vkvg_amd.Surface.from_bitmap(dev, b) for b in bitmaps]
        for signature in (True, False):
            s = vkvg_amd.Surface(dev, size, size, signature=signature)
            s.replay(sc.words(), srcs)
            assert np.array_equal(s.premultiplied(), rgba)
            if signature:
                assert np.array_equal(s.signature(), sig)
            s.close()
        for b in srcs:
            b.close()
