"""The front end at the sizes where its kernels change hands: scan tables around the
length of one workgroup's scan, tile rows beyond the table that adds up a workgroup's
entries, and contours of fewer, as many and more cubics than lanes share a path."""
import numpy as np
import pytest

import tileink_amd as tk

from test_gpu_frontend import CubicScene, PolygonScene, assert_same_scene, check_move, scene_arrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,count", [
    (2048, 2048, 30),     # 16384 tiles: the longest table of one workgroup
    (2064, 2048, 30),     # 16512: three launches for the tiles, one for the rest
    (200, 150, 16380),    # the paths about as many
    (200, 150, 16600),
    (40, 65536, 40),      # 4096 tile rows, a canvas's most and the table's
])
def test_table_sizes_rebuild_the_host_encoding(ctx, width, height, count):
    sc = PolygonScene(width + count, width, height, count=count, occluders=2, clips=count < 100)
    frame = tk.Frame(ctx, sc.record(sc.polygons).encode(0))
    check_move(ctx, sc, frame, sc.moved(3, scale=1.2))


def test_a_batch_of_more_tile_rows_than_the_table(ctx):
    scenes = [PolygonScene(60 + i, 40, 36000, count=25) for i in range(2)]  # 2250 rows each
    batch = tk.Batch(ctx, [s.record(s.polygons).encode(0) for s in scenes])
    moved = [s.moved(70 + i, scale=1.5) for i, s in enumerate(scenes)]
    parts = [s.points(m) for s, m in zip(scenes, moved)]
    starts = np.concatenate([parts[0][1][:-1], parts[1][1] + len(parts[0][0])]).astype(np.uint32)
    batch.frame.set_polygons(np.concatenate([p for p, _ in parts]), starts)
    ref = tk.Batch(ctx, [s.record(m).encode(0) for s, m in zip(scenes, moved)])
    assert_same_scene(scene_arrays(batch.frame), scene_arrays(ref.frame))
    batch.render()
    ref.render()
    for i in range(2):
        assert np.array_equal(batch.image(i), ref.image(i)), i


def test_contours_of_any_number_of_cubics_flatten_like_the_recorder(ctx):
    sc = CubicScene(5, 320, 240)
    rng = np.random.default_rng(12)
    sc.contours, sc.ops = [], []
    for n in (1, 2, 7, 8, 9, 15, 16, 17, 40, 3):
        k = sc._contour(rng, *rng.uniform(40, 200, 2), 150.0, n)
        sc.ops.append(("path", k, (0.2, 0.1 * (n % 9), 0.7, 0.6), n % 2))
    frame = tk.Frame(ctx, sc.record(sc.contours).encode(0))
    for contours in (sc.contours, sc.moved(9)):
        frame.set_cubic_paths(*sc.ctrl(contours), tolerance=0.25)
        ref = tk.Frame(ctx, sc.record(contours).encode(0))
        assert_same_scene(scene_arrays(frame), scene_arrays(ref))
        frame.render()
        ref.render()
        assert np.array_equal(frame.image(), ref.image())


@pytest.mark.parametrize("paths", [11264, 11265])  # the flattener's table alone: one workgroup, three launches
def test_flattened_tables_of_either_scan(ctx, paths):
    rng = np.random.default_rng(paths)
    ctrl = rng.uniform(2, 118, (paths, 1, 2)) + rng.uniform(-4, 4, (paths, 7, 2))
    ctrl[:, 6] = ctrl[:, 0]
    ctrl[::5, 3] = ctrl[::5, 0]  # curves of another number of lines

    def record():
        canvas = tk.Canvas(120, 120)
        for c in ctrl:
            path = tk.BezPath().move_to(*c[0]).curve_to(*c[1:4].reshape(-1)).curve_to(*c[4:7].reshape(-1))
            canvas.push_path(path.close_path(), tk.Color(0.3, 0.6, 0.2, 0.1))
        return canvas.encode(0)

    scene = record()
    frame = tk.Frame(ctx, scene)
    want = scene_arrays(frame)
    ctrl += 1.0
    frame.set_cubic_paths(ctrl.reshape(-1, 2), np.arange(paths + 1, dtype=np.uint32) * 7)
    ctrl -= 1.0
    frame.set_cubic_paths(ctrl.reshape(-1, 2), np.arange(paths + 1, dtype=np.uint32) * 7)
    assert_same_scene(scene_arrays(frame), want)
