"""The one-kernel scan of scenes laid out path by path (tk_k_path_scan): runs of
small paths, paths at the edges of a run's tables, large paths shared out by tile
rows, and the scenes it leaves to the separate stages, all against the oracle."""
import numpy as np
import pytest

import tileink_amd as tk
from tileink_amd import _abi

import oracle

from helpers import channel_diff, compare_frame, read_frame, tile_sorted_segments

pytestmark = pytest.mark.gpu

RUN = 928      # lines, tiles and paths (four each) per run, at most (TK_PATH_SCAN_RUN)
LINES = 8192   # lines from which a path in a small frame is long
MOST = 64512   # lines of the longest path it takes (TK_PATH_SCAN_LINES)


def _pays(arrays):
    """path_scan_rule.h: whether the one-kernel scan is the faster for a scene."""
    lines, tiles, visits = (arrays.paths[:, k].astype(np.int64) for k in (1, 5, 11))
    reach = np.minimum(3 * tiles, 1024 * visits // np.maximum(lines, 1))
    even = 4096 + lines + reach
    most = len(arrays.lines) // 256 + int(np.where(tiles > 1280, reach, 0).max()) // 3
    worst = max(0, (visits - even).max(), (lines - 6144 - np.minimum(2 * tiles, 2048)).max())
    shared = np.where(tiles > 1280, tiles // 640 * (8192 + lines + visits), 0).sum()
    return bool(worst <= most and shared <= (1 << 27) + 12 * len(arrays.lines))


def _swapped(arrays):
    """The scene with two lines of different paths exchanged, which the one-kernel scan refuses."""
    out = tk.SceneArrays.__new__(tk.SceneArrays)
    out.__dict__.update(arrays.__dict__)
    out.lines = arrays.lines.copy()
    ids = arrays.lines["path_id"]
    k = int(np.nonzero(ids[1:] != ids[:-1])[0][0])
    out.lines[[k, k + 1]] = arrays.lines[[k + 1, k]]
    return out


def _box(canvas, x0, y0, tiles_x, tiles_y, rng):
    """A concave polygon whose tile box is tiles_x by tiles_y tiles from (x0, y0)."""
    w, h = 16 * tiles_x - 2, 16 * tiles_y - 2
    mid = rng.uniform(0.2, 0.8, 2)
    path = tk.BezPath().move_to(16 * x0 + 1, 16 * y0 + 1)
    for u, v in ((1, 0), (mid[0], mid[1]), (1, 1), (0, 1)):
        path.line_to(16 * x0 + 1 + u * w, 16 * y0 + 1 + v * h)
    canvas.push_path(path.close_path(), tk.Color(*rng.uniform(0, 1, 3), 0.5), rule=tk.FillRule(int(rng.integers(2))))


def _zigzag(canvas, lines, width, height, rng):
    """One path of exactly `lines` lines."""
    pts = rng.uniform((0.0, 0.0), (width, height), (lines, 2))
    path = tk.BezPath().move_to(*pts[0])
    for p in pts[1:]:
        path.line_to(*p)
    canvas.push_path(path.close_path(), tk.Color(0.2, 0.6, 0.9, 0.5), rule=tk.FillRule.EvenOdd)


def _matches(ctx, canvas, one=True):
    gpu, ref, bad = compare_frame(ctx, canvas)
    assert not bad, (bad, channel_diff(gpu["image"], ref["image"]))
    assert gpu["stats"]["one_kernel_scan"] == one


# tile boxes on canvases little larger, in runs of 128 or the canvas's width: single
# tiles, two runs' tiles and one more (the first size that is shared out), past three,
# many bands of uneven rows, and the widest canvas
@pytest.mark.parametrize("tiles", [(1, 1), (16, 16), (1, 256), (1, 257), (20, 13), (16, 24), (35, 11), (128, 2), (131, 67),
                                   (RUN - 2, 4)])
def test_path_sizes_match_oracle(ctx, tiles):
    rng = np.random.default_rng(tiles[0])
    tw, th = max(tiles[0] + 2, 20), max(tiles[1] + 2, 12)
    canvas = tk.Canvas(16 * tw, 16 * th)
    for k in range(5):
        for _ in range(40):
            _box(canvas, int(rng.integers(0, 15)), int(rng.integers(0, 8)), *rng.integers(1, 5, 2), rng)
        _box(canvas, 0, k % 2, *tiles, rng)
        canvas.push_path(tk.BezPath().move_to(-90, 5).line_to(-20, 9).line_to(-30, 40).close_path(), tk.Color(1, 0, 0, 1))
    _matches(ctx, canvas)


def test_shared_rows_meet_lines_that_leave_the_canvas(ctx):
    rng = np.random.default_rng(5)
    canvas = tk.Canvas(1500, 1100)
    for k in range(6):
        path = tk.BezPath().move_to(*rng.uniform(-900, 2400, 2))
        for _ in range(12):
            path.line_to(*rng.uniform(-900, 2400, 2))
        canvas.push_path(path.close_path(), tk.Color(*rng.uniform(0, 1, 3), 0.4), rule=tk.FillRule(k % 2))
        canvas.push_stroke(path, 7.0, tk.Color(0, 0.3 * (k % 3), 1, 0.6))
    _matches(ctx, canvas)


@pytest.mark.parametrize("lines,width,height", [(LINES, 200, 200), (LINES + 1, 200, 200), (300, 16 * (RUN + 1), 64)])
def test_long_and_wide_paths_match_oracle(ctx, lines, width, height):
    rng = np.random.default_rng(lines)
    canvas = tk.Canvas(width, height)
    _zigzag(canvas, 50, width, height, rng)
    _zigzag(canvas, lines, width, height, rng)
    _zigzag(canvas, 30, width, height, rng)
    _matches(ctx, canvas, one=False)


def test_lines_within_one_tile_match_the_general_traversal(ctx):
    """Short lines, which skip the traversal: ends on tile corners and edges, level
    lines on and off a tile's top, lines a hair long, at every side of the canvas."""
    rng = np.random.default_rng(3)
    canvas = tk.Canvas(100, 70)
    for k in range(300):
        at = rng.choice([0.0, 16.0, 32.0, 48.0, 63.9999, 64.0, 95.0, 96.0, 100.0], 2) * (1.0, 0.7)
        path = tk.BezPath().move_to(*at)
        for _ in range(int(rng.integers(2, 9))):
            step = rng.choice([0.0, 1e-6, 1e-3, 0.5, 3.0, 15.9999, 16.0], 2) * rng.choice([-1.0, 1.0], 2)
            at = at + step
            path.line_to(*at)
        canvas.push_path(path.close_path(), tk.Color(*rng.uniform(0, 1, 3), 0.5), rule=tk.FillRule(k % 2))
    _matches(ctx, canvas)


def _mixed_canvas():
    rng = np.random.default_rng(11)
    canvas = tk.Canvas(1300, 900)
    for k in range(60):
        if k % 20 == 7:
            _zigzag(canvas, 40, 1300, 900, rng)
        _box(canvas, int(rng.integers(0, 70)), int(rng.integers(0, 45)), *rng.integers(1, 12, 2), rng)
    return canvas


def test_lines_in_another_order_give_the_same_frame(ctx):
    """Lines that do not lie path by path go through the separate stages, to the same
    tables, segments and image; an update changes the route of a frame."""
    arrays = _mixed_canvas().arrays(0)
    shuffled = tk.SceneArrays.__new__(tk.SceneArrays)
    shuffled.__dict__.update(arrays.__dict__)
    shuffled.lines = arrays.lines[np.random.default_rng(1).permutation(len(arrays.lines))].copy()
    scenes = [arrays.to_scene(), shuffled.to_scene()]
    frame = tk.Frame(ctx, scenes[0])
    frame.set_capture(True)
    first = None
    for k in (0, 1, 0):
        scene = scenes[k]
        frame.update(scene)
        frame.render()
        out = read_frame(frame, scene)
        assert out["stats"]["one_kernel_scan"] == (k == 0)
        if first is None:
            first = out
        for key in ("raw_backdrops", "backdrops", "segment_counts", "segment_ranges", "segment_cursors", "segment_bumps",
                    "tile_ptcl_counts", "tile_kinds", "ptcl", "image"):
            assert np.array_equal(out[key], first[key]), key
        assert np.array_equal(tile_sorted_segments(out["segments"], out["segment_ranges"]),
                              tile_sorted_segments(first["segments"], first["segment_ranges"]))
    assert np.array_equal(first["image"], oracle.render_frame(arrays)[0])


def test_incremental_render_and_graph_replay_of_shared_rows(ctx):
    canvas = _mixed_canvas()
    scene = canvas.encode(0)
    want = oracle.render_frame(canvas.arrays(0))[0]
    frame = tk.Frame(ctx, scene)
    assert frame.stats()["one_kernel_scan"] == 1
    frame.render()
    assert np.array_equal(frame.image(), want)
    T = scene.tiles_width * scene.tiles_height
    for part in (np.arange(0, T, 7), np.array([T - 1]), np.arange(T)):
        frame.render_tiles(part.astype(np.uint32))
        assert np.array_equal(frame.image(), want)
    frame.set_graph(True)
    for _ in range(3):
        frame.render()
        assert np.array_equal(frame.image(), want)


def _many_batches(width, height, clips):
    """Nothing but rectangles under a clip each, and two triangles: few runs, large tables."""
    rng = np.random.default_rng(clips)
    canvas = tk.Canvas(width, height)
    for _ in range(2):
        _zigzag(canvas, 3, width, height, rng)
    for _ in range(clips):
        x, y = rng.uniform(0, 0.8, 2) * (width, height)
        canvas.push_clip_sdf_rect_layer(x, y, x + 90, y + 60, 6.0)
        canvas.push_rect(x - 4, y, x + 70, y + 50, 8.0, tk.Color(*rng.uniform(0, 1, 3), 0.6))
        canvas.pop_layer()
        canvas.push_rect(x, y, x + 20, y + 20, 2.0, tk.Color(*rng.uniform(0, 1, 3), 1.0))
    return canvas


# tables cleared by the workgroups of the runs alone, by as many as their words ask for
# (4096 a workgroup), and by as many as there may be (2048)
@pytest.mark.parametrize("width,height,clips", [(48, 32, 3), (500, 300, 60), (4096, 4096, 70)])
def test_tables_of_many_batches_start_cleared(ctx, width, height, clips):
    arrays = _many_batches(width, height, clips).arrays(0)
    swapped = _swapped(arrays)  # the separate stages, whose tables are cleared in front
    frame = tk.Frame(ctx, arrays.to_scene())
    n = frame.batch_count * frame.tiles

    def tables():
        return [frame.image()] + [frame.buffer(b, np.uint32, n) for b in (_abi.BUF_TILE_PTCL_COUNTS, _abi.BUF_TILE_KINDS)]

    frame.render()
    assert frame.stats()["one_kernel_scan"] == 1
    first = tables()
    if n < 20000:
        assert np.array_equal(first[0], oracle.render_frame(arrays)[0])
    frame.update(swapped.to_scene())
    frame.render()
    assert frame.stats()["one_kernel_scan"] == 0
    for a, b in zip(first, tables()):
        assert np.array_equal(a, b)
    frame.update(arrays.to_scene())
    frame.render()
    for a, b in zip(first, tables()):
        assert np.array_equal(a, b)


# paths whose visits, lines or shares end what the rule allows, beside small ones: lines
# across one run's tiles, across shared ones, and lines of a visit each
@pytest.mark.parametrize("kind,lines,width,one", [
    ("across", 700, 120, True), ("across", 1100, 120, False), ("across", 250, 500, True), ("across", 900, 500, False),
    ("along", 5500, 120, True), ("along", 6600, 120, False), ("along", 8000, 600, True), ("along", 9900, 600, False),
    ("far", 5000, 1500, True), ("far", 11000, 1500, False),
])
def test_long_paths_take_the_route_of_the_rule(ctx, kind, lines, width, one):
    rng = np.random.default_rng(lines)
    canvas = tk.Canvas(width, width)
    _zigzag(canvas, 40, width, width, rng)
    if kind == "far":  # short lines in a corner, beside a path whose lines reach across
        _zigzag(canvas, 30, width, width, rng)
        pts = 60.0 * rng.uniform(size=(lines, 2)) + 2.0
    elif kind == "across":
        pts = rng.uniform(1.0, width - 1.0, (lines, 2))
    else:  # a curve of steps far shorter than a tile
        t = np.arange(lines) * 0.005
        pts = width * (0.5 + 0.48 * np.stack([np.cos(t), np.sin(1.3 * t)], 1))
    canvas.push_polygon(pts, tk.Color(0.7, 0.2, 0.4, 0.5), rule=tk.FillRule.EvenOdd)
    _box(canvas, 0, 0, 3, 3, rng)
    assert _pays(canvas.arrays(0)) == one
    _matches(ctx, canvas, one)


def test_many_shared_paths_leave_the_one_kernel_scan(ctx):
    # each shared by 102 workgroups, for 0.95 M of the 134 M that a sum may reach
    for count, one in ((135, True), (150, False)):
        canvas = tk.Canvas(4096, 4096)
        pts = np.array([[1, 1], [4095, 30], [4094, 4095], [3, 4090]], np.float64)
        canvas.push_polygons(np.tile(pts, (count, 1)), [4] * count, np.tile(np.float32([[0.2, 0.5, 0.9, 0.02]]), (count, 1)),
                             [0] * count)
        arrays = canvas.arrays(0)
        assert _pays(arrays) == one
        frame = tk.Frame(ctx, arrays.to_scene())
        frame.render()
        image, stats = frame.image(), frame.stats()
        assert stats["one_kernel_scan"] == one and stats["overflow"] == 0
        other = _swapped(arrays)
        frame.update(other.to_scene())
        frame.render()
        assert frame.stats()["one_kernel_scan"] == 0
        assert np.array_equal(frame.image(), image)


@pytest.mark.parametrize("lines", [MOST, MOST + 1])
def test_the_longest_path_beside_many_lines(ctx, lines):
    """In a frame of enough lines the longest path its queues can number is taken."""
    rng = np.random.default_rng(2)
    canvas = tk.Canvas(1024, 1024)
    n = 256 * (MOST - 6144 - 2048) // 24 + 100
    a = np.arange(24) * (2 * np.pi / 24)
    pts = rng.uniform(4, 1020, (n, 1, 2)) + 3.0 * np.stack([np.cos(a), np.sin(a)], 1)
    canvas.push_polygons(pts.reshape(-1, 2), np.full(n, 24), np.tile(np.float32([[0.3, 0.6, 0.1, 0.1]]), (n, 1)), np.zeros(n))
    walk = 512.0 + 300.0 * np.stack([np.cos(np.arange(lines) * 0.01), np.sin(np.arange(lines) * 0.013)], 1)
    canvas.push_polygon(walk, tk.Color(0.9, 0.1, 0.2, 0.7), rule=tk.FillRule.EvenOdd)
    arrays = canvas.arrays(0)
    assert _pays(arrays)
    frame = tk.Frame(ctx, arrays.to_scene())
    frame.render()
    stats, first = frame.stats(), None
    assert stats["one_kernel_scan"] == (lines == MOST) and stats["overflow"] == 0
    for scene in (arrays, _swapped(arrays)):
        frame.update(scene.to_scene())
        frame.render()
        out = [frame.image(), frame.buffer(_abi.BUF_BACKDROPS, np.int32, stats["backdrop_len"]),
               frame.buffer(_abi.BUF_SEGMENT_RANGES, np.uint32, 2 * stats["backdrop_len"])]
        first = first or out
        for x, y in zip(out, first):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("cubics", [False, True])
def test_moves_change_the_route_of_a_frame(ctx, graph, cubics):
    """The front end's side of the rule: a path that grows long and short again."""
    rng = np.random.default_rng(8)
    width = 200

    def geometry(long):
        if not cubics:
            polys = [rng.uniform(1, 60, (5, 2)), rng.uniform(1, width - 1, (long, 2)), rng.uniform(90, 180, (7, 2))]
        else:  # closed contours of cubics, of some eleven lines each
            polys = []
            for n in (2, long // 4, 3):
                p = rng.uniform(1, width - 1, (3 * n + 1, 2))
                p[-1] = p[0]
                polys.append(p)
        return polys

    def canvas_of(polys):
        canvas = tk.Canvas(width, width)
        for i, p in enumerate(polys):
            path = tk.BezPath().move_to(*p[0])
            if cubics:
                for k in range(1, len(p), 3):
                    path.curve_to(*p[k:k + 3].reshape(-1))
            else:
                for q in p[1:]:
                    path.line_to(*q)
            canvas.push_path(path.close_path(), tk.Color(0.2 * i, 0.5, 0.8, 0.6), rule=tk.FillRule(i % 2))
        return canvas

    def rounded(polys):
        return polys if cubics else [p.astype(np.float32).astype(np.float64) for p in polys]

    frame = tk.Frame(ctx, canvas_of(rounded(geometry(60))).encode(0))
    frame.set_graph(graph)
    for long, one in ((300, True), (2500, False), (240, True), (2000, False), (2000, False), (100, True)):
        polys = rounded(geometry(long))
        points = np.concatenate(polys)
        starts = np.concatenate([[0], np.cumsum([len(p) for p in polys])]).astype(np.uint32)
        if cubics:
            frame.set_cubic_paths(points, starts)
        else:
            frame.set_polygons(points.astype(np.float32), starts)
        arrays = canvas_of(polys).arrays(0)
        assert _pays(arrays) == one
        want = oracle.render_frame(arrays)[0]
        for _ in range(3 if graph else 1):
            frame.render()
            assert np.array_equal(frame.image(), want)
        assert frame.stats()["one_kernel_scan"] == one


@pytest.mark.parametrize("tiles", [RUN, RUN + 1])
def test_moves_on_the_widest_canvas(ctx, tiles):
    rng = np.random.default_rng(tiles)

    def polys():
        return [rng.uniform((1, 1), (16 * tiles - 1, 60), (n, 2)).astype(np.float32) for n in (5, 40, 12)]

    def canvas_of(ps):
        canvas = tk.Canvas(16 * tiles, 64)
        for p in ps:
            canvas.push_polygon(p.astype(np.float64), tk.Color(0.1, 0.7, 0.3, 0.5), rule=tk.FillRule.EvenOdd)
        return canvas

    frame = tk.Frame(ctx, canvas_of(polys()).encode(0))
    for _ in range(2):
        ps = polys()
        frame.set_polygons(np.concatenate(ps), np.concatenate([[0], np.cumsum([len(p) for p in ps])]).astype(np.uint32))
        frame.render()
        assert frame.stats()["one_kernel_scan"] == (tiles == RUN)
        assert np.array_equal(frame.image(), oracle.render_frame(canvas_of(ps).arrays(0))[0])


@pytest.mark.parametrize("scale,shift", [(1.0, (32.0, -48.0)), (2.0, (0.0, 0.0)), (0.5, (16.0, 7.5))])
def test_path_transforms_match_oracle(ctx, scale, shift):
    """Lines in a path's own space: every third path's, the others' transform the identity."""
    rng = np.random.default_rng(9)
    canvas = tk.Canvas(700, 500)
    for k in range(90):
        pts = np.round(rng.uniform(-40, 90, (6, 2)) * 8) / 8 + 16 * rng.integers(0, 36, 2)
        canvas.push_polygon(pts, tk.Color(*rng.uniform(0, 1, 3), 0.5), rule=tk.FillRule(k % 2))
    canvas.push_polygon(np.round(rng.uniform(0, 690, (30, 2))), tk.Color(0.1, 0.2, 0.8, 0.3), rule=tk.FillRule.EvenOdd)
    plain = canvas.arrays(0)
    moved = tk.SceneArrays.__new__(tk.SceneArrays)
    moved.__dict__.update(plain.__dict__)
    moved.lines, moved.paths = plain.lines.copy(), plain.paths.copy()
    own = np.arange(len(moved.paths)) % 3 == 0
    transform = np.array([scale, 0.0, 0.0, scale, *shift], np.float32)
    moved.paths[own, 13:19] = transform.view(np.uint32)
    mine = own[moved.lines["path_id"]]
    for end in ("p0", "p1"):  # exact: eighths of a pixel by powers of two
        moved.lines[end][mine] = (plain.lines[end][mine] - np.float32(shift)) / np.float32(scale)
    frame = tk.Frame(ctx, moved.to_scene())
    frame.render()
    assert frame.stats()["one_kernel_scan"] == 1
    want = oracle.render_frame(moved)[0]
    assert np.array_equal(want, oracle.render_frame(plain)[0])
    assert np.array_equal(frame.image(), want)
    other = _swapped(moved)
    frame.update(other.to_scene())
    frame.render()
    assert frame.stats()["one_kernel_scan"] == 0
    assert np.array_equal(frame.image(), want)
