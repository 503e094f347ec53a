"""Differentiable renderer at the edges of its row units against the FP64 reference: paths of one tile, of
exactly eight tiles and more (128 columns are added up at a time), across all borders of the image, edges
on tile borders, images smaller than a tile and paths off the image, and a stroke so wide and tight that its
parts lie over one another up to 14 times. And the coverage beside an outline, which has to cancel exactly.

Tolerances: coordinates below 512 are spaced 3e-5 px and an edge's ends take about four roundings, so an
edge lies within 1.2e-4 px of the reference's, which moves the coverage of a pixel by at most that per
edge in it, of which these scenes have up to four: 5e-4. Roundings are spread evenly over half a spacing
either way, 0.9e-5 in the mean square, 1.8e-5 for four of them: 2e-5 of the image's norm if an edge lay in every
pixel (measured: 0.02e-5). Colours' gradients add up one coverage per pixel, of which at most a quarter lie on an
edge: half of that, 1e-5 (measured: 0.4e-5). The gradients of control points and widths are integrals of numbers
known to 5e-4 over pieces known to that, and a pixel whose coverage lies within rounding of 1 counts or does not
count: 2e-3 of their norm (measured: 0.03e-3). The tight stroke's segments are 0.4 px long and 23 px from their
edges, where the roundings of a segment's ends, at coordinates spaced 8e-6, come to 4.5e-4 px, one for the whole
segment: four times the image's bounds (measured: 0.2e-5 of its norm), and 5e-4 for colours; its other gradients
are not compared, since single pixels of coverage near 1 decide them."""
import numpy as np
import pytest

from oracle import diff_ref as D

pytestmark = pytest.mark.gpu


def _polygon(points, bend=0.0):
    """A closed path of cubics through the points, straight (control points at thirds) or bent by that part
    of their length."""
    p = np.asarray(points, np.float64)
    d = np.roll(p, -1, 0) - p
    side = bend * d[:, ::-1] * [-1, 1]
    return np.stack([p, p + d / 3 + side, p + 2 * d / 3 + side], 1).reshape(-1, 2)


def _scene(name):
    r = np.random.Generator(np.random.PCG64(77))
    if name == "tile":  # within one tile, within two
        return 64, 48, [_polygon(16 + 14 * r.random((4, 2))), _polygon([20, 10] + 20 * r.random((3, 2)), 0.3)], [0, 1]
    if name == "aligned":  # borders on pixels, tiles and the 128 columns
        box = lambda x0, y0, x1, y1: _polygon([(x0, y0), (x1, y0), (x1, y1), (x0, y1)])  # noqa: E731
        return 288, 32, [box(16, 0, 144, 16), box(128, 5, 256, 32), box(0.5, 8, 128, 9), box(-20, 12, 300, 20)], [0] * 4
    if name == "wide":  # several times 128 columns, across all borders
        w = np.array([[-40.3, 7.7], [150.2, -9.1], [430.6, 22.3], [260.4, 61.8], [90.1, 44.4]])
        return 391, 40, [_polygon(w), _polygon(w[::-1] * [0.6, 0.8] + [30.5, 3.1]), _polygon(w * 0.9, 0.3)], [0, 0, 1]
    if name == "tall":
        w = np.array([[3.3, -20.7], [17.2, 80.1], [9.6, 200.3], [-6.4, 141.8]])
        return 15, 177, [_polygon(w), _polygon(w + [2.2, 9.3], 0.3)], [0, 1]
    if name == "tight":  # a loop of 12 px drawn 46 px wide: some of it is covered 14 times
        a = np.arange(6) * (2 * np.pi / 6)
        w = np.stack([90.3 + 6 * np.cos(a), 40.7 + 5 * np.sin(a)], 1)
        return 160, 80, [_polygon(w, 0.13), _polygon([[20, 20], [60, 12], [40, 66]], 0.2)], [46.0, 0]
    if name == "long":  # rows of 1300 edges and three times 128 columns, shared out over workgroups
        a = np.sort(r.uniform(0, 2 * np.pi, 170))
        w = np.stack([150 + 170 * np.cos(a), 18 + 13 * np.sin(a)], 1) + r.normal(0, 1, (170, 2))
        return 291, 37, [_polygon(w), _polygon([[20, 5], [60, 30], [99, 7]]), _polygon(w[::12] * [0.9, 1.1], 0.1)], [0, 0, 1]
    if name == "flat":  # edges across hundreds of columns in a row, and up to three times the 32 that a lane takes
        w = np.array([[-30.5, 3.3], [1480.2, 9.1], [700.7, 19.8]])
        return 1471, 23, [_polygon(w), _polygon(w[::-1] * [0.93, 0.8] + [30.5, 3.1]), _polygon(w * [0.3, 1], 0.01)], [0, 1, 1]
    if name == "point":  # one pixel, and a path that misses it on each side
        return 1, 1, [_polygon([[-0.7, 0.3], [0.6, -0.4], [0.9, 1.6]]), _polygon([[5, 5], [7, 5], [6, 8]]),
                      _polygon([[-9, 0.2], [-4, 0.4], [-6, 0.9]]), _polygon([[0.1, -8], [0.7, -3], [0.3, -5]])], [0, 0, 1, 0]
    paths = []
    for _ in range(12):  # "curved": closed cubics of all sizes
        c, s = r.uniform(0, (211, 75)), np.exp(r.uniform(0, 4.0))
        paths.append(c + s * r.standard_normal((3 * int(r.integers(1, 5)), 2)))
    return 211, 75, paths, list(r.integers(0, 2, 12))


@pytest.mark.parametrize("name", ["tile", "aligned", "wide", "tall", "tight", "long", "flat", "point", "curved"])
def test_rows_match_fp64_reference(name):
    import torch
    from vkvg_amd import diff
    W, H, paths, stroke = _scene(name)
    r = np.random.Generator(np.random.PCG64(5))
    n = len(paths)
    nc = np.array([len(p) // 3 for p in paths], np.uint32)
    wide = np.array(stroke, np.float32)  # a stroke's width where it is not 1
    stroke = (wide > 0).astype(np.uint32)
    ctrl = np.concatenate(paths).astype(np.float32)
    rgba = r.uniform(0.2, 0.9, (n, 4)).astype(np.float32)
    lw = np.where(wide > 1, wide, np.where(stroke, r.uniform(1, 5, n), 0)).astype(np.float32)
    g_img = r.standard_normal((H, W, 4)).astype(np.float32)
    ref_scene = D.Scene(W, H, nc, stroke)
    ref = D.forward(ref_scene, ctrl, rgba, lw)
    R = diff.DiffRenderer(W, H, nc, stroke)
    c, k, w = (torch.tensor(x, device="cuda") for x in (ctrl, rgba, lw))
    img = R.forward(c, k, w, keep=True)
    d = img.cpu().numpy() - ref
    print(name, "image", np.abs(d).max(), np.linalg.norm(d) / np.linalg.norm(ref), flush=True)
    f = 4 if name == "tight" else 1
    assert np.abs(d).max() < f * 5e-4 and np.linalg.norm(d) < f * 2e-5 * np.linalg.norm(ref)
    if name != "aligned":  # there |coverage| is exactly 1, where the clamp has no derivative
        g = torch.tensor(g_img, device="cuda")
        want = D.backward(ref_scene, ctrl, rgba, lw, g_img.astype(np.float64))
        for _ in range(2):  # a second backward of the same forward gives the same
            for what, a, b in zip(("ctrl", "rgba", "width"), R.backward(c, k, w, g), want):
                e = np.linalg.norm(a.cpu().numpy() - b) / max(np.linalg.norm(b), 1e-30)
                print(name, what, e, flush=True)
                if name == "tight":
                    assert what != "rgba" or e < 5e-4, (what, e)
                else:
                    assert e < (1e-5 if what == "rgba" else 2e-3), (what, e)
    assert np.abs(R.forward64(c, k, w).cpu().numpy() - ref).max() < 1e-9
    R.close()


@pytest.mark.parametrize("kind", ["blob", "wide", "star"])
def test_coverage_beside_an_outline_is_exact(kind):
    """Black opaque fills that wind around a point at most once: pixels that no edge comes near are exactly white
    outside (coverage 0, also between an outline's parts and right of it) and exactly black inside (coverage 1).
    Coordinates from 1 on are multiples of 2^-23, as every deposit is, so no sum up to 2 is rounded."""
    import torch
    from vkvg_amd import diff
    r = np.random.Generator(np.random.PCG64(19))
    W, H, m = {"blob": (150, 140, 40), "wide": (421, 60, 64), "star": (200, 190, 48)}[kind]
    for _ in range(8):
        a = np.sort(r.uniform(0, 2 * np.pi, m))
        rad = {"blob": 0.8 + 0.15 * np.sin(3 * a), "wide": 0.9 + 0.05 * np.cos(5 * a),
               "star": np.where(np.arange(m) % 2, 0.95, 0.45)}[kind]
        p = np.stack([W / 2 + 0.47 * W * rad * np.cos(a), H / 2 + 0.47 * H * rad * np.sin(a)], 1) + r.uniform(-0.3, 0.3, 2)
        ctrl = _polygon(p, 0.02).astype(np.float32)
        assert ctrl.min() >= 1
        nc, stroke = np.array([m], np.uint32), np.zeros(1, np.uint32)
        rgba, lw = np.array([[0, 0, 0, 1]], np.float32), np.zeros(1, np.float32)
        ref = D.forward(D.Scene(W, H, nc, stroke), ctrl, rgba, lw)[..., 0]
        edge = (ref > 1e-12) & (ref < 1 - 1e-12)
        near = np.zeros_like(edge)
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                near |= np.roll(edge, (dy, dx), (0, 1))
        R = diff.DiffRenderer(W, H, nc, stroke)
        img = R.forward(*(torch.tensor(x, device="cuda") for x in (ctrl, rgba, lw)))[..., 0].cpu().numpy()
        R.close()
        inside, outside = ~near & (ref < 0.5), ~near & (ref > 0.5)
        assert inside.sum() > 1000 and outside.sum() > 1000
        assert (img[outside] == 1).all() and (img[inside] == 0).all()


def test_a_path_in_few_rows_is_shared_out():
    """One path of 200 cubics over a strip of 8192x64 px: four tile rows of 64 times 128 columns and up to 3200 edges.
    With one workgroup per tile row its forward took 8.9 ms, with a lane per pixel row of an edge its backward 0.74."""
    import torch
    from vkvg_amd import diff
    r = np.random.Generator(np.random.PCG64(1))
    ctrl = (np.array([4096, 32]) + [2500, 20] * r.standard_normal((600, 2))).astype(np.float32)
    R = diff.DiffRenderer(8192, 64, np.array([200], np.uint32), np.zeros(1, np.uint32))
    args = [torch.tensor(x, device="cuda") for x in (ctrl, np.full((1, 4), 0.5, np.float32), np.zeros(1, np.float32))]
    ms = []
    for _ in range(5):
        img = R.forward(*args)
        ms.append(R.last_ms())
    bwd = []
    for _ in range(5):
        R.forward(*args, keep=True)
        R.backward(*args, torch.ones_like(img))
        bwd.append(R.last_ms(True))
    print(ms, bwd, flush=True)
    assert float((img.double() - R.forward64(*args)).abs().max()) < 2e-2  # coordinates of 8192 are spaced 1e-3
    R.close()
    assert min(ms) < 1.7 and min(bwd) < 0.4, (ms, bwd)


def test_more_row_units_than_a_launch_takes():
    """8200 paths over 1024 tile rows are 2^23 + 8192 workgroups: the last paths' rows are in a second launch."""
    import torch
    from vkvg_amd import diff
    n = 8200
    r = np.random.Generator(np.random.PCG64(2))
    one = np.array([[2, 4], [2, 16300], [14, 16380]], np.float32)  # a closed cubic from top to bottom
    ctrl = np.tile(one, (n, 1))
    rgba = np.concatenate([r.uniform(0, 1, (n, 3)), np.full((n, 1), 0.001)], 1).astype(np.float32)
    rgba[-1] = 0.25, 0.5, 0.75, 1
    nc, stroke = np.ones(n, np.uint32), np.zeros(n, np.uint32)
    img = []
    for k in (n, 1):  # all of them, and the last one alone
        R = diff.DiffRenderer(16, 16384, nc[-k:], stroke[-k:])
        args = [torch.tensor(x, device="cuda") for x in (ctrl[-3 * k:], rgba[-k:], np.zeros(k, np.float32))]
        img.append(R.forward(*args))
        R.close()
    inside = (img[1] - torch.tensor([0.25, 0.5, 0.75, 1.0], device="cuda")).abs().amax(-1) == 0
    assert int(inside.sum()) > 10000 and bool((img[0][inside] == img[1][inside]).all())
