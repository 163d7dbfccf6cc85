"""Coarse's chunks of 64 list entries: runs of batches that end, begin and go on at a
chunk's edge, batches whose layers act on some tiles only, and scenes of more layer
pairs than one tile holds in its lanes, against the oracle."""
import numpy as np
import pytest

import tileink_amd as tk

from helpers import channel_diff, compare_frame

pytestmark = pytest.mark.gpu


def _matches(ctx, canvas):
    gpu, ref, bad = compare_frame(ctx, canvas)
    assert not bad, (bad, channel_diff(gpu["image"], ref["image"]))


def _draw(canvas, rng, k):
    x, y = rng.uniform(-10, 110, 2)
    w, h = rng.uniform(4, 130, 2)
    color = tk.Color(*rng.uniform(0, 1, 3), 1.0 if k % 5 == 0 else 0.5)
    if k % 3 == 0:
        canvas.push_rect(x, y, x + w, y + h, float(rng.choice([0.0, 7.0])), color)
    else:
        path = tk.BezPath().move_to(x, y).line_to(x + w, y + 0.3 * h).line_to(x + 0.4 * w, y + h).close_path()
        canvas.push_path(path, color, rule=tk.FillRule(k % 2))


# entries of the runs a tile's list is made of: one run of a chunk and one more, runs
# that end on a chunk's edge, single entries, a run over three chunks
@pytest.mark.parametrize("runs", [(64,), (65,), (63, 1, 1), (64, 64), (1,) * 130, (10, 150, 3), (128, 64, 1)])
@pytest.mark.parametrize("partial", [False, True])
def test_runs_at_chunk_edges_match_oracle(ctx, runs, partial):
    rng = np.random.default_rng(len(runs) + 7 * runs[0])
    canvas = tk.Canvas(112, 96)
    for i, n in enumerate(runs):
        # a clip begins and ends a batch: around all tiles, or around some or none
        if i % 2:
            edge = float([30.0, 200.0, -20.0][i // 2 % 3]) if partial else -20.0
            canvas.push_clip_sdf_rect_layer(edge, edge, 140.0, 60.0 if partial and i % 4 == 3 else 140.0, 5.0)
        for k in range(n):
            # over the whole canvas, so that every tile lists every draw
            canvas.push_rect(-5.0, -5.0, 120.0, 110.0, 3.0, tk.Color(*rng.uniform(0, 1, 3), 0.3))
        if i % 2:
            canvas.pop_layer()
    _matches(ctx, canvas)


@pytest.mark.parametrize("pairs", [3, 64, 65, 90])
def test_scenes_of_many_layer_pairs_match_oracle(ctx, pairs):
    rng = np.random.default_rng(pairs)
    canvas = tk.Canvas(130, 110)
    for i in range(pairs):
        path = tk.BezPath().move_to(*rng.uniform(-20, 60, 2)).line_to(*rng.uniform(60, 150, 2)).line_to(0, 130).close_path()
        if i % 2:
            canvas.push_clip_layer(path, rule=tk.FillRule(i % 4 // 2))
        else:
            x, y = rng.uniform(-30, 40, 2)
            canvas.push_clip_sdf_rect_layer(x, y, x + 110, y + 100, 9.0)
        for k in range(3):
            _draw(canvas, rng, i + k)
        if i % 3:
            canvas.pop_layer()
            _draw(canvas, rng, i)
        elif i > 9:
            canvas.pop_layer()
    _matches(ctx, canvas)
