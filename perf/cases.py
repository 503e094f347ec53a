"""Timed cases of the renderer: what its users have it do, through its public entry points.

Raster frames go through the recorder and the frame pipeline in the four ways a program uses them:
"frame" (create a context on a surface, replay the drawing calls, destroy it: the frame is recorded,
uploaded and rendered), "readback" (the same, then the image in host memory as
vkvg_surface_write_to_memory returns it), "resident" (the frame uploaded once and executed again and
again, eagerly or as a captured graph) and "batch" (many surfaces in one submission). Their outputs
are bytes and have to stay the same. The differentiable renderer is timed forward and as a training
step (forward, L2 loss against a picture, backward to control points, colours and widths).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import vkvg_amd
from vkvg_amd import diff, scenes

_SHAPES = {"random": 6, "rounded": 2, "circles": 3, "stars": 5}


def listed() -> list[dict]:
    return [
        # a widget or an icon: a handful of shapes redrawn on every event; latency and launches
        dict(name="frame_shapes_256", path="frame", scene="shapes", size=256, n=16, shape="random"),
        # a page of a chart or a map with hundreds of filled and outlined shapes, odd-sized window
        dict(name="frame_shapes_777", path="frame", scene="shapes", size=777, n=500, shape="random"),
        # an illustration of large translucent curved fills rendered for an image file
        dict(name="readback_cubics_512", path="readback", scene="cubics", size=512, n=200),
        # a user interface: clips, save / restore, gradients, bitmaps as sources, operators, several
        # flushes, dashes and arcs interleaved
        dict(name="frame_mix_1021", path="frame", scene="mix", size=1021, n=300),
        # a drawing of thousands of small curved paths recorded and rendered once
        dict(name="frame_dense_1500", path="frame", scene="dense", size=1500, n=2500),
        # full-HD plots: long polylines with joins, caps and dashes, even-odd stars; drawn again per step
        dict(name="resident_strokes_1080p", path="resident", scene="strokes", width=1920, height=1080, n=7000,
             graph=False),
        # the dense 4K scene replayed as one captured graph
        dict(name="graph_dense_4096", path="resident", scene="dense", size=4096, n=20000, graph=True),
        # thumbnails: many uneven surfaces of strokes and stars rendered in one submission
        dict(name="batch_48", path="batch", scene="strokes", surfaces=48, side_lo=64, side_hi=1024, n_lo=10,
             n_hi=1000),
        # rendering parameters without a gradient (evaluation, line search)
        dict(name="diff_forward_512", path="diff", width=512, height=512, n=1024, train=False),
        # fitting a few paths to a thumbnail: latency of a small training step
        dict(name="diff_train_100x72", path="diff", width=100, height=72, n=48, train=True),
        # fitting paths to a picture, the usual size
        dict(name="diff_train_512", path="diff", width=512, height=512, n=1024, train=True),
        # a large picture with thousands of paths
        dict(name="diff_train_1024x768", path="diff", width=1024, height=768, n=3000, train=True),
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """One more case of the same ranges: sizes log-uniform, none costlier than the largest listed."""
    kind = rng.choice(["shapes", "cubics", "mix", "dense", "strokes", "batch", "diff", "diff"])
    if kind == "diff":
        w, h = _log(rng, 64, 1024), _log(rng, 64, 768)
        return dict(path="diff", width=w, height=h, n=_log(rng, max(4, w * h / 4096), max(8, w * h / 256)),
                    train=rng.random() < 0.75)
    if kind == "batch":
        hi = _log(rng, 128, 1024)
        return dict(path="batch", scene="strokes", surfaces=_log(rng, 4, 48), side_lo=64, side_hi=hi, n_lo=10,
                    n_hi=_log(rng, 40, 1000))
    path = rng.choice(["frame", "frame", "readback", "resident", "resident"])
    if kind == "mix" and path == "resident":  # surface sources and flushes are whole calls
        path = "frame"
    c = dict(path=path, scene=kind)
    if path == "resident":
        c["graph"] = rng.random() < 0.5
    if kind == "strokes":
        c.update(width=_log(rng, 200, 1920), height=_log(rng, 150, 1080), n=_log(rng, 30, 7000))
    else:
        size, n = {"shapes": ((64, 2048), (4, 3000)), "cubics": ((64, 1200), (4, 400)),
                   "mix": ((96, 1280), (20, 500)), "dense": ((256, 4096), (50, 20000))}[kind]
        c.update(size=_log(rng, *size), n=_log(rng, *n))
        if kind == "dense":
            # at most the density of the listed 4K scene
            c["n"] = max(20, min(c["n"], c["size"] * c["size"] * 20000 // (4096 * 4096)))
        if kind == "shapes":
            c["shape"] = rng.choice(sorted(_SHAPES))
    return c


# ------------------------------------------------------------------------------------ raster scenes
def _scene(case: dict, seed: int):
    """The case's drawing calls: (scene, bitmaps of its surface sources)."""
    kind, n = case["scene"], case["n"]
    if kind == "shapes":
        return scenes.randoms(_SHAPES[case["shape"]], "fill_stroke", n=n, size=case["size"], variant=seed), []
    if kind == "cubics":
        return scenes.config1(variant=seed, n_paths=n, size=case["size"]), []
    if kind == "mix":
        return scenes.grand_mix(variant=seed, size=case["size"], n=n)
    if kind == "dense":
        return scenes.config3(variant=seed, n_paths=n, size=case["size"]), []
    lines = max(1, n * 5 // 7)
    return scenes.config2(variant=seed, n_lines=lines, n_stars=n - lines, width=case["width"],
                          height=case["height"]), []


def _batch(case: dict, seed: int) -> list:
    """Square surfaces with sides and path counts log-uniform over the case's ranges (the same for
    every seed), each a drawing of strokes and stars."""
    g = np.random.Generator(np.random.PCG64(case["surfaces"]))
    sides = np.exp(g.uniform(math.log(case["side_lo"]), math.log(case["side_hi"]), case["surfaces"])).round()
    paths = np.exp(g.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]), case["surfaces"])).round()
    return [_scene(dict(scene="strokes", width=int(w), height=int(w), n=int(n)), 64 * seed + i)[0]
            for i, (w, n) in enumerate(zip(sides, paths))]


class _Owned:
    """A device or surface that is closed when nothing refers to it any more."""

    def __init__(self, obj, on=None):
        self.obj, self.on = obj, on  # `on`: the owner of the device that a surface lives on

    def __del__(self):
        self.obj.close()
        self.on = None


class _View:
    """A surface's image as a tensor without a copy; the tensor keeps the surface alive."""

    def __init__(self, owner):
        surf = owner.obj
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (surf.height, surf.width, 4), "typestr": "|u1", "version": 3,
                                         "data": (surf.device_ptr(), False), "strides": None}


_DEVICE = None


def _device():
    """The device a program creates once and draws every frame with."""
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = vkvg_amd.Device()
    return _DEVICE


class _Raster:
    def __init__(self, case: dict, seed: int):
        self.case, self.own, bitmaps = case, None, []
        dev = _device()
        if case["path"] == "batch":
            subs = _batch(case, seed)
            self.words = [s.words() for s in subs]
        else:
            sc, bitmaps = _scene(case, seed)
            subs, self.words = [sc], sc.words()
        if case["path"] == "resident":  # the resident frame belongs to its device
            self.own = _Owned(vkvg_amd.Device())
            dev = self.own.obj
            dev.set_graph(case["graph"])
        owners = [_Owned(vkvg_amd.Surface(dev, s.width, s.height), self.own) for s in subs]
        self.bitmaps = [_Owned(vkvg_amd.Surface.from_bitmap(dev, b), self.own) for b in bitmaps]
        self.surfs, self.sources = [o.obj for o in owners], [o.obj for o in self.bitmaps]
        self.images = [torch.as_tensor(_View(o), device="cuda") for o in owners]
        if case["path"] == "resident":
            self.surfs[0].upload(self.words)

    def run(self):
        path, surf = self.case["path"], self.surfs[0]
        if path == "batch":
            vkvg_amd.render_batch(_device(), self.surfs, self.words)
            return self.images
        if path == "resident":
            vkvg_amd.execute(self.own.obj)
            return self.images[0]
        surf.replay(self.words, self.sources)
        return surf.rgba() if path == "readback" else self.images[0]


# --------------------------------------------------------------------------- differentiable scenes
def _diff_inputs(case: dict, seed: int) -> dict:
    """Closed paths of 3..8 cubics around uniform centres, control points normal with s log-U[8, 64]
    (at most an eighth of the picture), half of them strokes of width U[1, 6]; the target is a smooth
    picture. The topology (cubics per path, which paths are strokes) is the same for every seed."""
    W, H, n = case["width"], case["height"], case["n"]
    g = np.random.Generator(np.random.PCG64(n))
    nc = g.integers(3, 9, n)
    stroke = g.random(n) < 0.5
    g = np.random.Generator(np.random.PCG64(seed))
    path = np.repeat(np.arange(n), 3 * nc)
    centre = np.stack([g.uniform(0, W, n), g.uniform(0, H, n)], 1)
    s = np.exp(g.uniform(math.log(8.0), math.log(max(9.0, min(64.0, max(W, H) / 8))), n))
    ctrl = centre[path] + s[path, None] * g.standard_normal((len(path), 2))
    rgba = np.concatenate([g.random((n, 3)), g.uniform(0.5, 1.0, (n, 1))], 1)
    width = np.where(stroke, g.uniform(1.0, 6.0, n), 0.0)
    coarse = torch.tensor(g.random((1, 4, 9, 9)))
    picture = torch.nn.functional.interpolate(coarse, size=(H, W), mode="bilinear", align_corners=True)
    f = np.float32
    return dict(ncubic=nc, stroke=stroke, ctrl=ctrl.astype(f), rgba=rgba.astype(f), width=width.astype(f),
                target=picture[0].permute(1, 2, 0).contiguous().float().numpy())


class _Diff:
    def __init__(self, case: dict, seed: int):
        d = _diff_inputs(case, seed)
        self.train = case["train"]
        self.scene = diff.DiffRenderer(case["width"], case["height"], d["ncubic"], d["stroke"])
        self.ctrl, self.rgba, self.width = (torch.tensor(d[k], device="cuda", requires_grad=self.train)
                                            for k in ("ctrl", "rgba", "width"))
        self.target = torch.tensor(d["target"], device="cuda")

    def run(self):
        img = diff.render(self.scene, self.ctrl, self.rgba, self.width)
        if not self.train:
            return img
        loss = ((img - self.target) ** 2).sum()
        gc, gr, gw = torch.autograd.grad(loss, (self.ctrl, self.rgba, self.width))
        return {"image": img.detach(), "ctrl": gc, "rgba": gr, "width": gw}


def prepare(case: dict, seed: int):
    return _Diff(case, seed) if case["path"] == "diff" else _Raster(case, seed)


def run(state):
    return state.run()


def work(case: dict) -> dict:
    """Bytes: the recorded calls (or the parameters and the picture) read once and the images written
    once. Operations: for a differentiable scene, some 20 per piece of an edge in a pixel row and
    pixel, about two pieces per edge and row; for a raster frame, one blend (16 operations) per pixel."""
    if case["path"] == "diff":
        W, H, n = case["width"], case["height"], case["n"]
        points = 5.5 * 16 * n
        data = 4 * (2 * 3 * 5.5 * n + 5 * n)
        pieces = 5.5 * points * 4
        if not case["train"]:
            return {"bytes": data + 16 * W * H, "flops": 20 * pieces + 8 * W * H}
        return {"bytes": 2 * data + 32 * W * H, "flops": 60 * pieces + 24 * W * H}
    subs = _batch(case, 0) if case["path"] == "batch" else [_scene(case, 0)[0]]
    px = sum(s.width * s.height for s in subs)
    return {"bytes": sum(s.words().nbytes for s in subs) + 4 * px, "flops": 16 * px}


def tolerance(case: dict):
    # Images are bytes. The differentiable renderer works in float32: its image differs from float64 by
    # up to 5.8e-6 (measured over the ranges). The gradient of a pixel's coverage jumps where the
    # covered area reaches 1, so rounding decides it at a few pixels: control points up to 1.6e-3,
    # widths 5.8e-4, colours 1e-6. About four times these.
    if case["path"] != "diff":
        return "exact"
    return {"rel": 6e-3 if case["train"] else 2e-5}


# ------------------------------------------------------------------------------- float64 reference
def _edges64(d: dict, ctrl, width):
    """Every path's edges in float64 (differentiable in ctrl and width): cubics sampled at i / 16;
    fills take the closed polyline, strokes per segment a rectangle and per vertex two bevel
    triangles of the same orientation."""
    dev = ctrl.device
    nc = d["ncubic"]
    first = np.concatenate([[0], np.cumsum(3 * nc)])
    path = np.repeat(np.arange(len(nc)), 16 * nc)
    j = np.concatenate([np.arange(16 * m) for m in nc])
    q, i = j // 16, j % 16
    t = torch.tensor(i / 16.0, device=dev)[:, None]
    u = 1 - t
    b = (u * u * u, 3 * u * u * t, 3 * u * t * t, t * t * t)
    pts = 0
    for k in range(4):
        idx = first[path] + (3 * q + k) % (3 * nc[path])
        pts = pts + b[k] * ctrl[torch.tensor(idx, device=dev)]
    start = np.concatenate([[0], np.cumsum(16 * nc)])
    p = np.arange(len(path))
    nxt = torch.tensor(np.where(j + 1 == 16 * nc[path], start[path], p + 1), device=dev)
    prv = torch.tensor(np.where(j == 0, start[path] + 16 * nc[path] - 1, p - 1), device=dev)
    stroke = torch.tensor(d["stroke"][path], device=dev)
    path = torch.tensor(path, device=dev)
    f = ~stroke
    out, owner = [torch.cat([pts[f], pts[nxt][f]], 1)], [path[f]]
    seg = pts[nxt] - pts
    nrm = torch.stack([-seg[:, 1], seg[:, 0]], 1) / seg.norm(dim=1, keepdim=True)
    off = (0.5 * width[path][:, None] * nrm)[stroke]
    off0 = (0.5 * width[path][:, None] * nrm[prv])[stroke]
    a, e, own = pts[stroke], pts[nxt][stroke], path[stroke]
    swap = (off0[:, 0] * off[:, 1] - off0[:, 1] * off[:, 0] > 0)[:, None]
    polys = [(a + off, e + off, e - off, a - off)]
    for s in (1.0, -1.0):
        v0, v1 = a + s * off0, a + s * off
        polys.append((a, torch.where(swap, v1, v0), torch.where(swap, v0, v1)))
    for poly in polys:
        for k, v in enumerate(poly):
            out.append(torch.cat([v, poly[(k + 1) % len(poly)]], 1))
            owner.append(own)
    edges, owner = torch.cat(out), torch.cat(owner)
    order = torch.argsort(owner, stable=True)
    return edges[order], owner[order]


def exact(case: dict, seed: int):
    """The differentiable renderer in plain float64: coverage is the integral of the winding number
    over a pixel, min(1, |.|) of it composited premultiplied source-over onto white; the coverage's
    derivative with respect to an edge is the boundary integral along the edge's part in the pixel.
    Raster frames: None (bytes, compared exactly)."""
    if case["path"] != "diff":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    d = _diff_inputs(case, seed)
    W, H, n, train = case["width"], case["height"], case["n"], case["train"]
    par = {k: torch.tensor(d[k], device=dev).double().requires_grad_(train) for k in ("ctrl", "rgba", "width")}
    target = torch.tensor(d["target"], device=dev).double()
    edges, owner = _edges64(d, par["ctrl"], par["width"])
    E = edges.detach()
    # (edge, pixel row) pairs
    lo, hi = torch.minimum(E[:, 1], E[:, 3]), torch.maximum(E[:, 1], E[:, 3])
    r0, r1 = lo.floor().clamp(0, H), hi.floor().clamp(-1, H - 1)
    cnt = torch.where(lo < hi, (r1 - r0 + 1).clamp(min=0), torch.zeros_like(lo)).long()
    pe = torch.repeat_interleave(torch.arange(len(E), device=dev), cnt)
    prow = r0[pe].long() + torch.arange(len(pe), device=dev) - (torch.cumsum(cnt, 0) - cnt)[pe]
    ppath = owner[pe]
    span = [0] + torch.cumsum(torch.bincount(ppath, minlength=n), 0).tolist()
    ax, ay, bx, by = E[pe].unbind(1)
    y0, y1 = torch.maximum(lo[pe], prow.double()), torch.minimum(hi[pe], prow.double() + 1)
    dx, dy = bx - ax, by - ay
    sa, sb = (y0 - ay) / dy, (y1 - ay) / dy
    s0, s1 = torch.minimum(sa, sb), torch.maximum(sa, sb)
    xa, xb = ax + s0 * dx, ax + s1 * dx
    xl, xr = torch.minimum(xa, xb), torch.maximum(xa, xb)
    area = torch.sign(dy) * (y1 - y0).clamp(min=0)
    box = torch.full((4, n), 1e9, device=dev, dtype=torch.float64)
    for k, v in enumerate((torch.minimum(E[:, 0], E[:, 2]), -torch.maximum(E[:, 0], E[:, 2]), lo, -hi)):
        box[k].scatter_reduce_(0, owner, v, "amin")
    box = box.cpu()
    cx0, cx1 = box[0].floor().clamp(0, W).int().tolist(), (-box[1]).floor().clamp(-1, W - 1).int().tolist()
    cy0, cy1 = box[2].floor().clamp(0, H).int().tolist(), (-box[3]).floor().clamp(-1, H - 1).int().tolist()
    col = par["rgba"].detach()
    pre = torch.cat([col[:, :3] * col[:, 3:], col[:, 3:]], 1)
    img = torch.ones((H, W, 4), device=dev, dtype=torch.float64)
    kept = []
    for p in range(n):
        if cx0[p] > cx1[p] or cy0[p] > cy1[p]:
            kept.append(None)
            continue
        s = slice(span[p], span[p + 1])
        X = torch.arange(cx0[p], cx1[p] + 2, device=dev, dtype=torch.float64)[None, :]
        l, r = xl[s, None], xr[s, None]
        left = torch.where(X >= r, X - 0.5 * (l + r), (X - l).clamp(min=0) ** 2 / (2 * (r - l).clamp(min=1e-300)))
        left = torch.where(X <= l, torch.zeros_like(left), left) * area[s, None]
        A = torch.zeros((cy1[p] - cy0[p] + 1, X.shape[1] - 1), device=dev, dtype=torch.float64)
        A.index_add_(0, prow[s] - cy0[p], left[:, 1:] - left[:, :-1])
        view = img[cy0[p]:cy1[p] + 1, cx0[p]:cx1[p] + 1]
        k = A.abs().clamp(max=1.0)[..., None]
        kept.append((A, view.clone()) if train else None)
        view.copy_(pre[p] * k + view * (1 - pre[p, 3] * k))
    if not train:
        return img
    g = 2 * (img - target)
    gE = torch.zeros_like(E)
    gcol = torch.zeros_like(col)
    for p in range(n - 1, -1, -1):
        if kept[p] is None:
            continue
        A, before = kept[p]
        gv = g[cy0[p]:cy1[p] + 1, cx0[p]:cx1[p] + 1]
        k = A.abs().clamp(max=1.0)[..., None]
        dk = (gv * (pre[p] - pre[p, 3] * before)).sum(-1)
        gp = (gv * k).sum((0, 1))
        gp[3] -= ((gv * before).sum(-1, keepdim=True) * k).sum()
        gcol[p, :3] = gp[:3] * col[p, 3]
        gcol[p, 3] = (gp[:3] * col[p, :3]).sum() + gp[3]
        gA = torch.where(A.abs() < 1, dk * torch.sign(A), torch.zeros_like(A))
        gv.mul_(1 - pre[p, 3] * k)
        s = slice(span[p], span[p + 1])
        X = torch.arange(cx0[p], cx1[p] + 2, device=dev, dtype=torch.float64)[None, :]
        safe = torch.where(dx[s] == 0, torch.ones_like(dx[s]), dx[s])[:, None]
        u = torch.minimum(torch.maximum((X - ax[s, None]) / safe, s0[s, None]), s1[s, None])
        up = torch.where(X > ax[s, None], s1[s, None], s0[s, None])  # vertical: all in one column
        u = torch.where(dx[s, None] == 0, up, u)
        q0, q1 = torch.minimum(u[:, :-1], u[:, 1:]), torch.maximum(u[:, :-1], u[:, 1:])
        i1 = 0.5 * (q1 * q1 - q0 * q0)
        rows = gA[prow[s] - cy0[p]]
        ga, gb = (rows * (q1 - q0 - i1)).sum(1), (rows * i1).sum(1)
        gE.index_add_(0, pe[s], torch.stack([-dy[s] * ga, dx[s] * ga, -dy[s] * gb, dx[s] * gb], 1))
    gc, gw = torch.autograd.grad(edges, (par["ctrl"], par["width"]), gE)
    return {"image": img, "ctrl": gc, "rgba": gcol, "width": gw}
