"""The calls a user of this framework makes, as timed cases.

A case is a dict of plain values.  Its `kind` says which entry point it goes
through; sizes, path counts, clip depths and options are its own.  The kinds:

  paths     tk.Frame(...).render(): cubic fills and strokes at the density of the
            benchmark's frame, solid and gradient paints, nested rounded-rectangle
            clips (`graph`: replayed from the frame's captured graph)
  polygons  tk.Frame(...).render(): solid polygons recorded in bulk
  mixed     tk.Frame(...).render(): a page of rectangles, fills, strokes, every
            brush kind, images, text outlines, path and rectangle clips
  tiles     Frame.render_tiles(...): the damaged block of a rendered frame again
  batch     tk.Batch(...).render(): independent canvases as one frame
  one_shot  NativeRenderer.render_to_image(canvas).readback(): canvas to host pixels
  animate   Frame.set_cubic_paths(...) + Frame.render(): the geometry moves, from
            control points on the GPU
  diff      diff.Plan forward + backward: FP32 image, line and colour gradients
  fit       diff.Renderer(...) + loss.backward(): parameters to their gradients

Images come back as the frame's own device pixels, gradients as the tensors the
calls return.  Rendered pixels are bytes and have to stay the same.
"""
import math

import numpy as np
import torch

import tileink_amd as tk
from tileink_amd import _abi, diff

_CONTEXT = []


def _context():
    """One context for the process, as a program keeps one."""
    if not _CONTEXT:
        _CONTEXT.append(tk.NativeContext(0))
    return _CONTEXT[0]


def listed():
    return [
        # One icon or glyph-sized canvas: the smallest call, all latency and launches.
        {"name": "icon", "kind": "paths", "width": 96, "height": 64, "paths": 24, "clips": 1, "graph": False},
        # A thumbnail redrawn every frame of a program's loop: launches replayed from the captured graph.
        {"name": "thumbnail_graph", "kind": "paths", "width": 333, "height": 257, "paths": 300, "clips": 2, "graph": True},
        # The parity workload's 640x360 canvas as one call from canvas to host pixels.
        {"name": "one_shot_640x360", "kind": "one_shot", "width": 640, "height": 360, "objects": 576},
        # A page or dashboard at screen size with every paint and primitive.
        {"name": "page_1920x1080", "kind": "mixed", "width": 1920, "height": 1080, "objects": 3000},
        # The benchmark's density and clip nesting at a quarter of its paths.
        {"name": "paths_2048_50k", "kind": "paths", "width": 2048, "height": 2048, "paths": 50000, "clips": 32,
         "graph": False},
        # A vector map: the benchmark's canvas and path count as polygons.
        {"name": "polygons_4096_200k", "kind": "polygons", "width": 4096, "height": 4096, "paths": 200000, "vertices": 24,
         "clips": 4},
        # An editor's redraw of the part that changed.
        {"name": "damage_1400x1000", "kind": "tiles", "width": 1400, "height": 1000, "paths": 12500, "clips": 8, "side": 16},
        # A renderer serving many canvases of ragged sizes at once.
        {"name": "batch_48", "kind": "batch", "scenes": 48, "low": 64, "high": 1024, "paths_mean": 400},
        # An animation: new control points every frame, flattened and binned on the GPU.
        {"name": "animate_1280x720", "kind": "animate", "width": 1280, "height": 720, "paths": 6000, "cubics": 6},
        # One differentiable scene, forward and backward, waiting for each call.
        {"name": "diff_256", "kind": "diff", "scenes": 1, "side": 256, "paths": 300, "sync": True, "keep": False},
        # The benchmark's batch of differentiable scenes at a quarter of its count, ordered on streams.
        {"name": "diff_batch_64x256", "kind": "diff", "scenes": 64, "side": 256, "paths": 288, "sync": False, "keep": False},
        # One optimiser step's forward and backward over a batch, from parameters to parameter gradients.
        {"name": "fit_32x200", "kind": "fit", "scenes": 32, "side": 200, "paths": 200},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["paths", "paths", "paths", "polygons", "mixed", "tiles", "batch", "one_shot", "animate", "diff", "diff",
                       "fit"])
    if kind == "paths":
        # up to the benchmark's density of about one path per 84 pixels
        w, h = _log(rng, 48, 2048), _log(rng, 48, 2048)
        return {"kind": kind, "width": w, "height": h, "paths": _log(rng, 10, max(20, w * h // 84)),
                "clips": rng.choice([0, 1, 2, 5, 12, 32]), "graph": rng.random() < 0.3}
    if kind == "polygons":
        w, h = _log(rng, 300, 4096), _log(rng, 300, 4096)
        return {"kind": kind, "width": w, "height": h, "paths": _log(rng, 200, max(400, w * h // 90)),
                "vertices": rng.randint(3, 24), "clips": rng.randint(0, 4)}
    if kind in ("mixed", "one_shot"):
        w, h = _log(rng, 150, 1920), _log(rng, 120, 1080)
        return {"kind": kind, "width": w, "height": h, "objects": _log(rng, 20, 3000 if kind == "mixed" else 600)}
    if kind == "tiles":
        w, h = _log(rng, 200, 1400), _log(rng, 200, 1000)
        return {"kind": kind, "width": w, "height": h, "paths": _log(rng, 200, max(400, w * h // 112)),
                "clips": rng.randint(0, 8), "side": rng.randint(1, 16)}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 48), "low": 64, "high": _log(rng, 128, 1024),
                "paths_mean": _log(rng, 50, 400)}
    if kind == "animate":
        return {"kind": kind, "width": _log(rng, 100, 1280), "height": _log(rng, 100, 720), "paths": _log(rng, 30, 6000),
                "cubics": rng.randint(3, 8)}
    if kind == "diff":
        return {"kind": kind, "scenes": _log(rng, 1, 64), "side": _log(rng, 48, 256), "paths": _log(rng, 20, 288),
                "sync": rng.random() < 0.5, "keep": rng.random() < 0.3}
    return {"kind": "fit", "scenes": _log(rng, 2, 32), "side": _log(rng, 48, 200), "paths": _log(rng, 20, 200)}


# --- recording ------------------------------------------------------------------------


class _Contour(tk.BezPath):
    """A path whose verb and point arrays are made already."""

    def __init__(self, verbs, points):
        self.verbs, self.points = verbs, points

    def arrays(self):
        return self.verbs, np.ascontiguousarray(self.points)


def _rng(seed, salt=0):
    return np.random.default_rng([0x71, int(seed), salt])


def _cubic_verbs(count, closed):
    return np.array([_abi.PATH_MOVE] + [_abi.PATH_CUBIC] * count + ([_abi.PATH_CLOSE] if closed else []), np.uint8)


_VERBS = {(k, c): _cubic_verbs(k, c) for k in range(1, 17) for c in (False, True)}


def _scribbles(rng, count, width, height, mu=math.log(48.0)):
    """Contours of 4-16 cubics with points uniform in a box of lognormal extent."""
    n = rng.integers(4, 17, count)
    size = 3 * n + 1
    first = np.concatenate([[0], np.cumsum(size)])
    extent = rng.lognormal(mu, 1.0, count)
    centre = rng.uniform(0.0, 1.0, (count, 2)) * (width, height)
    pts = rng.uniform(-0.5, 0.5, (int(first[-1]), 2)) * np.repeat(extent, size)[:, None] + np.repeat(centre, size, 0)
    return n.tolist(), first.tolist(), pts, centre, extent


def _colors(rng, count):
    c = rng.uniform(0.0, 1.0, (count, 4))
    c[:, 3] = 0.3 + 0.7 * c[:, 3]
    return c.tolist()


def _stops(rng):
    k = int(rng.integers(2, 5))
    offsets = np.sort(rng.uniform(0.0, 1.0, k))
    offsets[0], offsets[-1] = 0.0, 1.0
    return [(float(o), tk.Color(*c)) for o, c in zip(offsets, _colors(rng, k))]


def _linear(rng, centre, extent):
    a, b = centre + rng.uniform(-0.5, 0.5, 2) * extent, centre + rng.uniform(-0.5, 0.5, 2) * extent
    return tk.LinearGradient(tuple(a), tuple(b), _stops(rng), extend=int(rng.integers(0, 3)))


def _nested_clips(rng, canvas, box, depth, push):
    """Calls push(group) between `depth` nested clip layers going in and out."""
    box = np.asarray(box, np.float64)
    for g in range(2 * depth + 1):
        push(g)
        if g < depth:
            w, h = box[2] - box[0], box[3] - box[1]
            m = rng.uniform(0.0, 0.03, 4) * (w, h, w, h)
            box = box + (m[0], m[1], -m[2], -m[3])
            canvas.push_clip_sdf_rect_layer(*box, float(rng.uniform(0.0, min(64.0, 0.2 * w, 0.2 * h))))
        elif g < 2 * depth:
            canvas.pop_layer()


def _paths_canvas(rng, width, height, paths, clips):
    canvas = tk.Canvas(width, height)
    n, first, pts, centre, extent = _scribbles(rng, paths, width, height)
    fill = (rng.uniform(0, 1, paths) < 0.6).tolist()
    gradient = (rng.uniform(0, 1, paths) < 0.1).tolist()
    rules = rng.integers(0, 2, paths).tolist()
    widths = rng.lognormal(math.log(1.5), 0.7, paths).tolist()
    colors = _colors(rng, paths)
    groups = np.linspace(0, paths, 2 * clips + 2).astype(int)

    def push(g):
        for i in range(groups[g], groups[g + 1]):
            p = _Contour(_VERBS[n[i], fill[i]], pts[first[i]:first[i + 1]])
            brush = _linear(rng, centre[i], extent[i]) if gradient[i] else tk.Color(*colors[i])
            if fill[i]:
                p.points[-1] = p.points[0]
                canvas.push_path(p, brush, rule=tk.FillRule(rules[i]))
            else:
                canvas.push_stroke(p, widths[i], brush)

    _nested_clips(rng, canvas, (0.0, 0.0, width, height), clips, push)
    return canvas


def _polygons_canvas(rng, width, height, paths, vertices, clips):
    canvas = tk.Canvas(width, height)
    counts = rng.integers(3, vertices + 1, paths)
    first = np.concatenate([[0], np.cumsum(counts)])
    k = np.arange(int(first[-1])) - np.repeat(first[:-1], counts)
    angle = 2.0 * math.pi * k / np.repeat(counts, counts) + np.repeat(rng.uniform(0, 6.28, paths), counts)
    radius = np.repeat(np.minimum(rng.lognormal(math.log(14.0), 0.9, paths), 256.0), counts) * rng.uniform(0.5, 1.2, len(k))
    centre = np.repeat(rng.uniform(0.0, 1.0, (paths, 2)) * (width, height), counts, 0)
    pts = centre + radius[:, None] * np.stack([np.cos(angle), np.sin(angle)], 1)
    colors = np.asarray(_colors(rng, paths), np.float32)
    rules = rng.integers(0, 2, paths)
    groups = np.linspace(0, paths, 2 * clips + 2).astype(int)

    def push(g):
        lo, hi = groups[g], groups[g + 1]
        if hi > lo:
            canvas.push_polygons(pts[first[lo]:first[hi]], counts[lo:hi], colors[lo:hi], rules[lo:hi])

    _nested_clips(rng, canvas, (0.0, 0.0, width, height), clips, push)
    return canvas


def _picture(rng, height, width):
    y, x = np.mgrid[0:height, 0:width]
    rgba = np.stack([127.5 + 127.5 * np.sin(x * rng.uniform(0.05, 0.3) + y * rng.uniform(0.05, 0.3) + rng.uniform(0, 6))
                     for _ in range(4)], -1) + rng.normal(0, 10, (height, width, 4))
    return tk.Image.from_rgba8(np.clip(np.rint(rgba), 0, 255).astype(np.uint8))


def _blob(rng, centre, radius, cubics):
    """A smooth closed contour: ends on a jittered circle, tangent control points."""
    a = np.arange(cubics) * (2 * math.pi / cubics) + rng.uniform(0, 6.28)
    r = radius * rng.uniform(0.6, 1.2, cubics)
    ends = centre + r[:, None] * np.stack([np.cos(a), np.sin(a)], 1)
    k = 4.0 / 3.0 * math.tan(math.pi / (2 * cubics))
    tangent = r[:, None] * np.stack([-np.sin(a), np.cos(a)], 1)
    c1 = np.roll(ends + k * tangent, 1, 0)
    c2 = ends - k * tangent
    pts = np.concatenate([ends[-1:], np.stack([c1, c2, ends], 1).reshape(-1, 2)])
    return _Contour(_VERBS[cubics, True], pts)


def _mixed_canvas(rng, width, height, objects):
    canvas = tk.Canvas(width, height)
    size = np.array([width, height], np.float64)
    canvas.push_rect(0.0, 0.0, width, height, 0.0, tk.Color(0.97, 0.97, 0.95, 1.0))
    images = [canvas.add_image(_picture(rng, 48, 64)), canvas.add_image(_picture(rng, 24, 24))]

    def brush(c, e):
        kind = int(rng.integers(0, 12))
        if kind == 0:
            return _linear(rng, c, e)
        if kind == 1:
            return tk.RadialGradient(tuple(c), 0.0, tuple(c + rng.uniform(-0.1, 0.1, 2) * e), float(0.6 * e), _stops(rng),
                                     extend=int(rng.integers(0, 3)))
        if kind == 2:
            return tk.SweepGradient(tuple(c), 0.0, 2 * math.pi, _stops(rng))
        if kind == 3:
            return tk.FourCornerGradient((c[0] - e / 2, c[1] - e / 2, c[0] + e / 2, c[1] + e / 2),
                                         [tk.Color(*v) for v in _colors(rng, 4)])
        if kind == 4:
            s, a = 1.0 / max(e, 4.0), float(rng.uniform(0, 6.28))
            return tk.ImageBrush(images[int(rng.integers(0, 2))], (s * math.cos(a), -s * math.sin(a), s * math.sin(a),
                                                                   s * math.cos(a), 0.1, 0.2),
                                 extend=int(rng.integers(0, 3)), sampling=int(rng.integers(0, 2)))
        c4 = _colors(rng, 1)[0]
        return tk.Color(*c4[:3], 1.0 if rng.uniform() < 0.5 else c4[3])

    open_layers = 0
    for i in range(objects):
        c = rng.uniform(0.0, 1.0, 2) * size
        e = float(min(rng.lognormal(math.log(40.0), 0.8), 400.0))
        what = int(rng.integers(0, 20))
        if what < 7:
            w, h = e * rng.uniform(0.4, 2.0), e * rng.uniform(0.2, 1.0)
            canvas.push_rect(c[0] - w / 2, c[1] - h / 2, c[0] + w / 2, c[1] + h / 2, float(rng.uniform(0.0, 12.0)), brush(c, e))
        elif what < 12:
            canvas.push_path(_blob(rng, c, e / 2, int(rng.integers(3, 9))), brush(c, e), rule=tk.FillRule(int(rng.integers(0, 2))))
        elif what < 16:
            n = int(rng.integers(1, 5))
            canvas.push_stroke(_Contour(_VERBS[n, False], c + rng.uniform(-0.5, 0.5, (3 * n + 1, 2)) * e),
                               float(rng.lognormal(math.log(2.0), 0.5)), brush(c, e))
        elif what < 18:
            canvas.push_text_outline(_blob(rng, c, 7.0, int(rng.integers(4, 9))), tk.Color(0.1, 0.1, 0.15, 1.0))
        elif what < 19:
            canvas.push_image(c[0], c[1], c[0] + e, c[1] + 0.7 * e, images[0], extend=0, sampling=int(rng.integers(0, 2)))
        elif open_layers < 3:
            if rng.uniform() < 0.5:
                canvas.push_clip_layer(_blob(rng, size / 2, 0.55 * float(size.min()), 6))
            else:
                canvas.push_clip_sdf_rect_layer(0.03 * width, 0.04 * height, 0.96 * width, 0.95 * height, 18.0)
            open_layers += 1
        else:
            for _ in range(open_layers):
                canvas.pop_layer()
            open_layers = 0
    for _ in range(open_layers):
        canvas.pop_layer()
    return canvas


# --- differentiable scenes --------------------------------------------------------------


def _diff_inputs(seed, index, side, paths):
    """One scene's parameters as arrays: smooth closed contours of 4 cubics, straight
    colours, one clip, a tenth of the paints gradients of 2-4 stops."""
    rng = _rng(seed, 100 + index)
    n = paths
    a = np.arange(4)[None] * (math.pi / 2) + rng.uniform(0, 6.28, (n, 1))
    r = np.clip(rng.lognormal(math.log(16.0), 0.5, n), 4.0, 128.0)[:, None] * rng.uniform(0.6, 1.2, (n, 4))
    ends = rng.uniform(0, side, (n, 1, 2)) + r[..., None] * np.stack([np.cos(a), np.sin(a)], -1)
    k = 4.0 / 3.0 * math.tan(math.pi / 8.0)
    tangent = r[..., None] * np.stack([-np.sin(a), np.cos(a)], -1)
    c1 = np.roll(ends + k * tangent, 1, 1) + rng.normal(0, 1.0, ends.shape)
    c2 = ends - k * tangent + rng.normal(0, 1.0, ends.shape)
    fills = np.stack([c1, c2, ends], 2)
    colors = np.concatenate([rng.uniform(0, 1, (n, 3)), rng.uniform(0.3, 0.9, (n, 1))], 1)
    inset = rng.uniform(0.02, 0.1, 4) * side
    clip = (inset[0], inset[1], side - inset[2], side - inset[3], float(rng.uniform(2, 12)))
    gradients = {}
    for j, d in enumerate(np.sort(rng.permutation(n)[:n // 10])):
        s = 2 + j % 3
        x0, y0 = rng.uniform(0, side, 2)
        t, length = rng.uniform(0, 6.28), rng.uniform(16, 96)
        offsets = np.sort(rng.uniform(0, 1, s))
        offsets[0], offsets[-1] = 0.0, 1.0
        stops = np.concatenate([rng.uniform(0, 1, (s, 3)), rng.uniform(0.3, 1.0, (s, 1))], 1)
        gradients[int(d)] = ((x0, y0, x0 + length * math.cos(t), y0 + length * math.sin(t)), offsets,
                             stops.astype(np.float32), "radial" if rng.uniform() < 0.5 else "linear")
    return {"fills": fills.astype(np.float32), "colors": colors.astype(np.float32), "clip": clip,
            "rules": rng.integers(0, 2, n), "gradients": gradients}


def _diff_scene(p, side, device):
    t = lambda a: torch.tensor(a, dtype=torch.float32, device=device)
    s = diff.DiffScene(side, side, fills=t(p["fills"]), colors=t(p["colors"]), rules=p["rules"],
                       clips=[(*p["clip"], 0, len(p["rules"]))])
    s.gradients = {d: (line, off, t(stops), kind) for d, (line, off, stops, kind) in p["gradients"].items()}
    return s


_STEPS = 7  # the diff cases' polygons: chords per cubic


def _flatten(fills, steps=None):
    """Vertices of closed cubic contours cut at t = k / n, and vertices per contour; n is
    `steps`, or from the chord error bound 0.75 * max second difference <= 0.25 n^2
    (at most 256)."""
    ends = fills[:, :, 2]
    cub = torch.stack([torch.roll(ends, 1, 1), fills[:, :, 0], fills[:, :, 1], ends], 2).reshape(-1, 4, 2)
    p = cub.detach().double()
    a, b = p[:, 0] - 2 * p[:, 1] + p[:, 2], p[:, 1] - 2 * p[:, 2] + p[:, 3]
    dd = torch.maximum((a * a).sum(1).sqrt(), (b * b).sum(1).sqrt())
    n = torch.clamp(torch.ceil(torch.sqrt(0.75 * dd / 0.25)), 1, 256).long()
    if steps is not None:
        n = torch.full_like(n, steps)
    which = torch.repeat_interleave(torch.arange(len(n), device=n.device), n)
    k = torch.arange(int(n.sum()), device=n.device) - torch.repeat_interleave(torch.cumsum(n, 0) - n, n)
    t = (k.to(cub) / n[which].to(cub))[:, None]
    c = cub[which]
    v = (1 - t) ** 3 * c[:, 0] + 3 * t * (1 - t) ** 2 * c[:, 1] + 3 * t * t * (1 - t) * c[:, 2] + t ** 3 * c[:, 3]
    return v, n.reshape(fills.shape[0], -1).sum(1)


def _weights(seed, pixels, device):
    """dL/d(image) of the diff cases, a fixed field."""
    g = torch.Generator(device="cpu").manual_seed(int(seed) & 0x7FFFFFFF)
    return torch.randn((pixels, 4), generator=g).to(device)


def _target(seed, pixels, device):
    g = torch.Generator(device="cpu").manual_seed((int(seed) + 7) & 0x7FFFFFFF)
    return torch.rand((pixels, 4), generator=g).to(device)


# --- the cases --------------------------------------------------------------------------


class _Pixels:
    """A frame's device image as an array interface (one word per pixel)."""

    def __init__(self, address, words, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (words,), "typestr": "<i4", "data": (address, False), "version": 3,
                                         "strides": None}


def _device_words(frame, words, owner):
    """The frame's pixels in place; the tensor keeps `owner`, which frees them, alive."""
    return torch.as_tensor(_Pixels(int(_abi.lib().tk_frame_image_device(frame._h)), words, owner), device="cuda")


def _frame_state(canvas):
    frame = tk.Frame(_context(), canvas.encode(0))
    return {"frame": frame, "image": _device_words(frame, frame.width * frame.height, frame).view(frame.height, frame.width)}


def prepare(case, seed):
    kind, rng = case["kind"], _rng(seed)
    if kind == "paths":
        st = _frame_state(_paths_canvas(rng, case["width"], case["height"], case["paths"], case["clips"]))
        st["frame"].set_graph(case["graph"])
    elif kind == "polygons":
        st = _frame_state(_polygons_canvas(rng, case["width"], case["height"], case["paths"], case["vertices"], case["clips"]))
    elif kind == "mixed":
        st = _frame_state(_mixed_canvas(rng, case["width"], case["height"], case["objects"]))
    elif kind == "tiles":
        st = _frame_state(_paths_canvas(rng, case["width"], case["height"], case["paths"], case["clips"]))
        st["frame"].render()
        tw, th = (case["width"] + 15) // 16, (case["height"] + 15) // 16
        side = min(case["side"], tw, th)
        x0, y0 = int(rng.integers(0, tw - side + 1)), int(rng.integers(0, th - side + 1))
        st["tiles"] = (np.arange(y0, y0 + side)[:, None] * tw + np.arange(x0, x0 + side)).reshape(-1).astype(np.uint32)
    elif kind == "batch":
        canvases = []
        sizes = np.random.default_rng([case["scenes"], case["high"], case["paths_mean"]])  # the canvases, any contents
        for i in range(case["scenes"]):
            side = math.exp(sizes.uniform(math.log(case["low"]), math.log(case["high"])))
            aspect = math.sqrt(sizes.uniform(0.5, 2.0))
            n = int(np.clip(sizes.lognormal(math.log(case["paths_mean"]), 1.0), 10, 4 * case["paths_mean"]))
            canvases.append(_paths_canvas(_rng(seed, 1 + i), max(16, int(side * aspect)), max(16, int(side / aspect)), n,
                                          min(32, max(1, n // 256))))
        scenes = [c.encode(0) for c in canvases]
        batch = tk.Batch(_context(), scenes)
        columns = np.concatenate([[0], np.cumsum([s.tiles_width * s.tiles_height for s in scenes])])
        words = _device_words(batch.frame, int(columns[-1]) * 256, batch)
        st = {"batch": batch, "image": [words[c * 256:c * 256 + s.width * s.height].view(s.height, s.width)
                                        for s, c in zip(scenes, columns)]}
    elif kind == "one_shot":
        canvas = _mixed_canvas(rng, case["width"], case["height"], case["objects"])
        st = {"renderer": tk.NativeRenderer(tk.NativeBackend.Hip, case["width"], case["height"], context=_context()),
              "canvas": canvas}
    elif kind == "animate":
        n, cubics = case["paths"], case["cubics"]
        size = np.array([case["width"], case["height"]], np.float64)
        centres = rng.uniform(0, 1, (n, 2)) * size
        radii = np.minimum(rng.lognormal(math.log(18.0), 0.6, n), 200.0)
        colors = _colors(rng, n)
        blobs = [_blob(rng, c, r, cubics) for c, r in zip(centres, radii)]
        canvas = tk.Canvas(case["width"], case["height"])
        for b, c in zip(blobs, colors):
            canvas.push_path(b, tk.Color(*c))
        st = _frame_state(canvas)
        pts = np.concatenate([b.points for b in blobs])
        moved = pts + rng.normal(0, 4.0, pts.shape)
        first = np.arange(n) * (3 * cubics + 1)
        moved[first + 3 * cubics] = moved[first]
        st["ctrl"] = torch.as_tensor(moved, device="cuda")
        st["starts"] = torch.as_tensor(np.arange(n + 1) * (3 * cubics + 1), dtype=torch.int32, device="cuda")
    else:
        scenes = [_diff_scene(_diff_inputs(seed, i, case["side"], case["paths"]), case["side"], "cuda")
                  for i in range(case["scenes"])]
        if kind == "diff":
            polys = [_flatten(s.fills, _STEPS) for s in scenes]
            plan = diff.Plan(_context(), scenes, [v for v, _ in polys], [k.cpu().numpy() for _, k in polys],
                             sync=case["sync"])
            plan.frame.set_tuning(diff_keep_coverage=int(case["keep"]))
            paint = plan.full_paint(torch.cat([s.paint_records() for s in scenes]))
            st = {"plan": plan, "paint": paint, "grad": _weights(seed, plan.pixels, "cuda")}
        else:
            # every scene's parameters are slices of three tensors, as an optimiser holds a batch
            leaves = {"fills": torch.cat([s.fills for s in scenes]), "colors": torch.cat([s.colors for s in scenes])}
            grads = [(s, d) for s in scenes for d in sorted(s.gradients)]
            if grads:
                leaves["stops"] = torch.cat([s.gradients[d][2] for s, d in grads])
            for t in leaves.values():
                t.requires_grad_(True)
            at = 0
            for i, s in enumerate(scenes):
                n = case["paths"]
                s.fills, s.colors = leaves["fills"][i * n:(i + 1) * n], leaves["colors"][i * n:(i + 1) * n]
                for d in sorted(s.gradients):
                    line, off, stops, k = s.gradients[d]
                    s.gradients[d] = (line, off, leaves["stops"][at:at + len(off)], k)
                    at += len(off)
            renderer = diff.Renderer(_context(), scenes, "cuda", sync=False)
            renderer()  # records the scenes; later calls move their vertices
            st = {"renderer": renderer, "leaves": leaves, "target": _target(seed, renderer.flat.shape[0], "cuda")}
    torch.cuda.synchronize()
    return st


def run(state):
    if "batch" in state:
        state["batch"].render()
        return state["image"]
    if "canvas" in state:
        return state["renderer"].render_to_image(state["canvas"]).readback()
    if "plan" in state:
        image = state["plan"].forward(state["paint"])
        line_grad, color_grad = state["plan"].backward(state["grad"])
        return {"image": image, "line_grad": line_grad, "color_grad": color_grad}
    if "leaves" in state:
        renderer, leaves = state["renderer"], state["leaves"]
        for t in leaves.values():
            t.grad = None
        renderer()
        flat = renderer.flat
        ((flat - state["target"]) ** 2).sum().backward()
        return {"image": flat.detach(), **{k: t.grad for k, t in leaves.items()}}
    frame = state["frame"]
    if "ctrl" in state:
        frame.set_cubic_paths(state["ctrl"], state["starts"])
        frame.render()
    elif "tiles" in state:
        frame.render_tiles(state["tiles"])
    else:
        frame.render()
    return state["image"]


# Lines a path of each generator flattens to, and tiles its boundary meets, on average.
_LINES = {"paths": 227.0, "mixed": 40.0}


def work(case):
    """Bytes: the scene's lines (24 B), path and draw records (200 B) and paint (80 B)
    in, the pixels out; a differentiable pass reads the geometry again, reads one
    gradient image and writes line and colour gradients.  Operations: 40 per line
    for its tile walk and row coverage, 12 per covered pixel for its blend."""
    kind = case["kind"]
    if kind in ("paths", "tiles", "polygons", "mixed", "one_shot", "animate"):
        pixels = case["width"] * case["height"]
        if kind in ("mixed", "one_shot"):
            n, lines, area = case["objects"], _LINES["mixed"], 1600.0
        elif kind == "polygons":
            n, lines, area = case["paths"], 0.5 * (3 + case["vertices"]), 900.0
        elif kind == "animate":
            n, lines, area = case["paths"], 5.0 * case["cubics"], 1400.0
        else:
            n, lines, area = case["paths"], _LINES["paths"], 2500.0
        share = 1.0
        if kind == "tiles":
            tiles = ((case["width"] + 15) // 16) * ((case["height"] + 15) // 16)
            share = min(1.0, case["side"] ** 2 / tiles)
        return {"bytes": share * (n * (24 * lines + 280) + 4 * pixels), "flops": share * n * (40 * lines + 12 * area)}
    if kind == "batch":
        n = case["scenes"] * 1.3 * case["paths_mean"]
        mean = (case["high"] ** 2 - case["low"] ** 2) / (2 * math.log(case["high"] / case["low"]))
        return {"bytes": n * (24 * _LINES["paths"] + 280) + 4 * case["scenes"] * mean,
                "flops": n * (40 * _LINES["paths"] + 12 * 2000.0)}
    n, lines, pixels = case["scenes"] * case["paths"], 28.0, case["scenes"] * case["side"] ** 2
    more = 2 if kind == "fit" else 1
    return {"bytes": n * (24 * lines + 16 * lines + 280 + 256) * more + 48 * pixels,
            "flops": n * (3 * 40 * lines + 40 * 700.0)}


def tolerance(case):
    """Rendered pixels are bytes: the same.  The differentiable form composites in
    FP32 over up to 300 layers and sums its gradients in FP32 in no fixed order: it
    is within 1e-6 of 64 bits (2-norm), and its parameter gradients, through
    vertices evaluated in FP32, within 1.5e-5."""
    if case["kind"] == "diff":
        return {"rel": 4e-6, "max": 1e-3}
    if case["kind"] == "fit":
        return {"rel": 5e-5, "max": 2e-3}
    return "exact"


# --- the differentiable form in 64 bits ---------------------------------------------------


def _pieces64(a, b, width, height):
    """Lines a -> b cut at every pixel boundary inside the canvas: (line, s0, s1, row,
    column) of each piece, s the line's parameter.  A piece left of the canvas is
    given column -1, one right of it `width`."""
    def crossings(p, q, limit):
        lo = torch.clamp(torch.floor(torch.minimum(p, q)) + 1, 0, limit + 1)
        hi = torch.clamp(torch.ceil(torch.maximum(p, q)) - 1, -1, limit)
        count = torch.clamp(hi - lo + 1, min=0).long()
        line = torch.repeat_interleave(torch.arange(len(p), device=p.device), count)
        k = torch.arange(len(line), device=p.device) - torch.repeat_interleave(torch.cumsum(count, 0) - count, count)
        return line, (lo[line] + k - p[line]) / (q - p)[line]

    lines = torch.arange(len(a), device=a.device)
    lx, sx = crossings(a[:, 0], b[:, 0], width)
    ly, sy = crossings(a[:, 1], b[:, 1], height)
    line = torch.cat([lines, lines, lx, ly])
    s = torch.cat([torch.zeros(len(a), device=a.device, dtype=a.dtype), torch.ones(len(a), device=a.device, dtype=a.dtype),
                   sx.clamp(0, 1), sy.clamp(0, 1)])
    order = torch.argsort(s)
    order = order[torch.argsort(line[order], stable=True)]
    line, s = line[order], s[order]
    same = line[1:] == line[:-1]
    line, s0, s1 = line[:-1][same], s[:-1][same], s[1:][same]
    mid = a[line] + (0.5 * (s0 + s1))[:, None] * (b - a)[line]
    row, col = torch.floor(mid[:, 1]).long(), torch.floor(mid[:, 0]).long()
    ok = (row >= 0) & (row < height)
    return line[ok], s0[ok], s1[ok], row[ok], col[ok].clamp(-1, width)


def _exact_scene(p, side, steps, weights=None, target=None):
    """FP64 image, dL/d(lines) and dL/d(paint) of one scene, and dL/d(parameters)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t64 = lambda x: torch.as_tensor(x, dtype=torch.float64, device=dev)
    n = len(p["rules"])
    fills = t64(p["fills"]).requires_grad_(True)
    colors = t64(p["colors"]).requires_grad_(True)
    verts, counts = _flatten(fills, steps)
    if steps is None:
        v = verts.detach().float().double()  # the vertices are stored in 32 bits
    else:  # the polygons that the plan was given
        v = _flatten(torch.as_tensor(p["fills"], device=dev), steps)[0].double()
    start = torch.cumsum(counts, 0) - counts
    path = torch.repeat_interleave(torch.arange(n, device=dev), counts)
    nxt = torch.arange(len(v), device=dev) + 1
    nxt = torch.where(nxt == (start + counts)[path], start[path], nxt)
    a, b = v, v[nxt]
    line, s0, s1, row, col = _pieces64(a, b, side, side)
    d = (b - a)[line]
    dy = d[:, 1] * (s1 - s0)
    xm = a[line, 0] + 0.5 * (s0 + s1) * d[:, 0]
    diffs = torch.zeros((n, side, side + 1), dtype=torch.float64, device=dev)
    at = (path[line] * side + row) * (side + 1)
    inside = (col >= 0) & (col < side)
    left = torch.where(inside, 1.0 - (xm - col), torch.ones_like(xm))  # share of the piece's own pixel
    first = col.clamp(0, side)
    diffs.view(-1).index_add_(0, at + first, -dy * left)
    rest = inside
    diffs.view(-1).index_add_(0, (at + first + 1)[rest], (-dy * (1.0 - left))[rest])
    cov = torch.cumsum(diffs, 2)[:, :, :side].contiguous().requires_grad_(True)
    y, x = torch.meshgrid(torch.arange(side, device=dev) + 0.5, torch.arange(side, device=dev) + 0.5, indexing="ij")
    x, y = x.double(), y.double()
    x0, y0, x1, y1, radius = p["clip"]
    # the clip's rectangle and radius are stored in 32 bits
    x0, y0, x1, y1, radius = (float(np.float32(c)) for c in (x0, y0, x1, y1, radius))
    hx, hy = 0.5 * (x1 - x0), 0.5 * (y1 - y0)
    r = max(min(radius, hx, hy), 0.0)
    qx, qy = (x - 0.5 * (x0 + x1)).abs() - hx + r, (y - 0.5 * (y0 + y1)).abs() - hy + r
    dist = torch.maximum(qx, qy).clamp(max=0) + torch.sqrt(qx.clamp(min=0) ** 2 + qy.clamp(min=0) ** 2) - r
    mask = (0.5 - dist).clamp(0, 1)
    pm = torch.cat([colors[:, :3] * colors[:, 3:], colors[:, 3:]], 1)
    records = {}
    stop_leaves = []
    image = torch.zeros((side, side, 4), dtype=torch.float64, device=dev)
    paints = []
    for i in range(n):
        w = cov[i]
        alpha = (w - 2 * torch.round(0.5 * w.detach())).abs() if p["rules"][i] else w.abs().clamp(max=1.0)
        alpha = (alpha * mask)[..., None]
        if i in p["gradients"]:
            (gx0, gy0, gx1, gy1), off, stops, kind = p["gradients"][i]
            gx0, gy0, gx1, gy1 = (float(np.float32(c)) for c in (gx0, gy0, gx1, gy1))
            off = [float(np.float32(o)) for o in off]
            leaf = t64(stops).requires_grad_(True)
            stop_leaves.append(leaf)
            spm = torch.cat([leaf[:, :3] * leaf[:, 3:], leaf[:, 3:]], 1)
            gdx, gdy = gx1 - gx0, gy1 - gy0
            den = gdx * gdx + gdy * gdy
            if kind == "radial":
                t = torch.sqrt(((x - gx0) ** 2 + (y - gy0) ** 2) / den)
            else:
                t = ((x - gx0) * gdx + (y - gy0) * gdy) / den
            t = t.clamp(0, 1)
            ws = torch.zeros((len(off), side, side), dtype=torch.float64, device=dev)
            ws[0] += (t <= off[0]).double()
            for j in range(len(off) - 1):
                if off[j + 1] > off[j]:
                    u = (t - off[j]) / (off[j + 1] - off[j])
                    here = ((t > off[j]) & (t < off[j + 1])).double()
                    ws[j] += here * (1 - u)
                    ws[j + 1] += here * u
            ws[-1] += ((t >= off[-1]) & (t > off[0])).double()
            for j in range(1, len(off) - 1):
                ws[j] += ((t == off[j]) & (t > off[0])).double()
            color = (ws[..., None] * spm[:, None, None, :]).sum(0)
            paints.append(spm)
        else:
            color = pm[i]
            paints.append(color[None] if color.dim() == 1 else color)
        paints[-1].retain_grad()
        if i not in p["gradients"]:
            color = paints[-1][0]
        image = image * (1 - alpha * color[..., 3:]) + alpha * color
    flat = image.reshape(-1, 4)
    if weights is not None:
        loss = (flat * weights.to(flat)).sum()
    else:
        loss = ((flat - target.to(flat)) ** 2).sum()
    loss.backward(retain_graph=True)
    # a line moves the coverage of the pixels it crosses along its normal
    g = cov.grad[path[line], row, col.clamp(0, side - 1)] * inside
    i1 = 0.5 * (s1 * s1 - s0 * s0)
    g0 = torch.zeros(len(a), dtype=torch.float64, device=dev).index_add_(0, line, g * ((s1 - s0) - i1))
    g1 = torch.zeros(len(a), dtype=torch.float64, device=dev).index_add_(0, line, g * i1)
    nx, ny = a[:, 1] - b[:, 1], b[:, 0] - a[:, 0]
    line_grad = torch.stack([-nx * g0, -ny * g0, -nx * g1, -ny * g1], 1)
    # the clip's own draw comes first, with no paint of its own
    color_grad = torch.zeros((n + 1, 32), dtype=torch.float64, device=dev)
    for i, q in enumerate(paints):
        color_grad[i + 1, 16:16 + 4 * len(q)] = q.grad.reshape(-1)
    gv = torch.zeros_like(v).index_add_(0, torch.arange(len(v), device=dev), line_grad[:, :2])
    gv.index_add_(0, nxt, line_grad[:, 2:])
    verts.backward(gv)
    return {"image": flat.detach(), "line_grad": line_grad, "color_grad": color_grad, "fills": fills.grad,
            "colors": colors.grad, "stops": [s.grad for s in stop_leaves]}


def exact(case, seed):
    """The differentiable cases in FP64; rendered pixels are bytes and need none."""
    if case["kind"] not in ("diff", "fit") or case["scenes"] * case["paths"] > 8000:
        return None
    side = case["side"]
    columns = ((side + 15) // 16) ** 2
    pixels = side * side if case["scenes"] == 1 else case["scenes"] * columns * 256
    make = _weights if case["kind"] == "diff" else _target
    field = make(seed, pixels, "cpu")
    flat, parts = torch.zeros((pixels, 4), dtype=torch.float64), []
    for i in range(case["scenes"]):
        at = i * columns * 256
        f = field[at:at + side * side].to("cuda" if torch.cuda.is_available() else "cpu")
        p = _exact_scene(_diff_inputs(seed, i, side, case["paths"]), side, _STEPS if case["kind"] == "diff" else None,
                         **({"weights": f} if case["kind"] == "diff" else {"target": f}))
        flat[at:at + side * side] = p["image"].cpu()
        parts.append({k: [s.cpu() for s in v] if k == "stops" else v.cpu() for k, v in p.items() if k != "image"})
    join = lambda k: torch.cat([q[k] for q in parts])
    if case["kind"] == "diff":
        return {"image": flat, "line_grad": join("line_grad"), "color_grad": join("color_grad")}
    out = {"image": flat, "fills": join("fills"), "colors": join("colors")}
    stops = [s for q in parts for s in q["stops"]]
    if stops:
        out["stops"] = torch.cat(stops)
    return out
