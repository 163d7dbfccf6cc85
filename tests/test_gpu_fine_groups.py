"""Fine builds coverage four records at a time, eight lanes to a segment, over
windows of 64 records that run across a tile's batches: the sizes where a group, a
window or a pass over the segments ends, and segments no scan emits, against the
per-pixel coverage entry and the oracle."""
import ctypes as C

import numpy as np
import pytest

import tileink_amd as tk
from tileink_amd import _abi
from tileink_amd._abi import check, lib

from helpers import compare_frame

pytestmark = pytest.mark.gpu

INTERPRETER, END, FILL = 0, 0, 1


def _segments(rng, n, kind):
    p = rng.uniform(0, 16, (n, 4)).astype(np.float32)
    if kind == "short":  # a flattened curve's
        p[:, 2:] = np.clip(p[:, :2] + rng.normal(0, 2.0, (n, 2)), 0, 16)
    elif kind == "boundary":  # ends on and beside pixel boundaries
        p = np.round(p) + rng.choice([0, 1e-6, -1e-6, 2.0 ** -20], (n, 4))
    elif kind == "powers":  # widths one unit below a power of two, and tiny ones
        p[:, 0] = rng.choice([2.0 ** -37, 2.0 ** -26, 1e-30, 0.0, 2.0 ** -70], n)
        p[:, 2] = np.nextafter(np.float32(2.0) ** rng.integers(0, 5, n), np.float32(0))
        p[:, 1] = np.floor(p[:, 1])
        p[:, 3] = p[:, 1] + rng.choice([1.0, 0.5, 16.0], n)
    elif kind == "outside":  # what no scan emits
        p = rng.choice([np.nan, np.inf, -np.inf, -5.5, 40.25, 0.0, 16.0, 7.25, 1e30], (n, 4))
    edge = np.where(rng.uniform(size=n) < 0.3, rng.uniform(-2, 18, n), 1e9)
    if kind == "outside":
        edge = rng.choice([np.nan, -np.inf, np.inf, -3.0, 0.0, 15.999, 16.0, 1e9], n)
    return np.concatenate([p, edge[:, None]], 1).astype(np.float32)


@pytest.mark.parametrize("kind", ["short", "boundary", "powers", "outside"])
@pytest.mark.parametrize("rule", [0, 1])
def test_grouped_coverage_equals_the_per_pixel_sums(ctx, kind, rule):
    rng = np.random.default_rng(len(kind) + rule)
    counts = [0, 1, 7, 8, 9, 31, 32, 33, 64, 65, 200]
    before = [0, 1, 2, 3, 4, 5, 62, 63, 64, 65, 130]  # records ahead of the one under test
    tiles = [(n, k) for n in counts for k in before]
    segs, ptcl, ranges, requests = [], [], [], []
    at = 0
    for t, (n, k) in enumerate(tiles):
        start = len(ptcl)
        for i in range(k):  # transparent fills: they draw nothing, their segments are summed
            m = int(rng.integers(0, 12))
            segs.append(_segments(rng, m, "short"))
            ptcl.append((FILL, 0, i & 1, at, at + m, 1))
            at += m
        backdrop = int(rng.integers(-2, 3))
        segs.append(_segments(rng, n, kind))
        ptcl.append((FILL, backdrop, rule, at, at + n, 0))
        requests += [(at, at + n, np.int32(backdrop).view(np.uint32), x, y, rule, 0, 0)
                     for y in range(16) for x in range(16)]
        at += n
        ptcl.append((END, 0, 0, 0, 0, 0))
        ptcl += [(FILL, 1, 0, 0, at, 0)] * (t % 3)  # past END: never drawn
        ranges.append((start, len(ptcl)))
    segs = np.concatenate(segs) if at else np.zeros((1, 5), np.float32)
    T = len(tiles)
    draws = np.zeros((2, 31), np.uint32)
    record = np.zeros(2, np.dtype(_abi.DrawRecord))
    record["brush_offset"] = [0, 16]
    record["sdf_offset"] = record["sdf_shadow_offset"] = _abi.INVALID
    draws[:] = record.view(np.uint32).reshape(2, 31)
    paint = np.zeros(32, np.uint32)
    paint[0], paint[4] = _abi.BRUSH_SOLID, 0xFFFFFFFF
    paint[16], paint[20] = _abi.BRUSH_SOLID, 0x00000000
    cfg = _abi.FineConfig(16 * T, 16, 0, T, T, 1, 1, 0, 32, 0, 0, 2, len(ptcl), len(segs))
    keep = [ctx.to_device(a) for a in (draws, paint, segs, np.array(ranges, np.uint32),
                                       np.full(T, INTERPRETER, np.uint32), np.array(ptcl, np.int64).astype(np.uint32))]
    d_draws, d_paint, d_segs, d_ranges, d_kinds, d_ptcl = keep
    inputs = _abi.FineInputs()
    inputs.draws, inputs.paint, inputs.segments = d_draws.ptr, d_paint.ptr, d_segs.ptr
    inputs.tile_ptcl_ranges, inputs.tile_kinds, inputs.ptcl = d_ranges.ptr, d_kinds.ptr, d_ptcl.ptr
    rgba = ctx.to_device(np.zeros(256 * T, np.uint32))
    check(lib().tk_fine(ctx.handle, C.byref(cfg), C.byref(inputs), rgba.ptr))
    req = ctx.to_device(np.array(requests, np.uint32))
    alpha = ctx.to_device(np.zeros(256 * T, np.uint32))
    check(lib().tk_fill_coverage_words(ctx.handle, 256 * T, req.ptr, d_segs.ptr, alpha.ptr, None))
    ctx.synchronize()
    # opaque white over nothing: every channel is the record's alpha
    got = rgba.read(np.uint32).reshape(16, T, 16).transpose(1, 0, 2).reshape(-1)
    want = alpha.read(np.uint32) * np.uint32(0x01010101)
    bad = np.nonzero(got != want)[0]
    assert bad.size == 0, [(tiles[b // 256], b % 256, hex(got[b]), hex(want[b])) for b in bad[:5]]


@pytest.mark.parametrize("groups,fills", [(1, 1), (1, 4), (1, 5), (1, 63), (1, 64), (1, 65), (3, 2), (33, 1), (33, 3)])
def test_streams_across_batches_match_oracle(ctx, groups, fills):
    # `groups` draw groups under nested clips: 2 * (groups // 2) + 1 batches of short
    # streams on every tile, so windows and groups run across batches.
    rng = np.random.default_rng(100 * groups + fills)
    canvas = tk.Canvas(70, 50)
    depth = groups // 2

    def draw():
        for _ in range(fills):
            path = tk.BezPath().move_to(*rng.uniform(-5, 75, 2))
            for _ in range(3):
                path.curve_to(*rng.uniform(-5, 75, 6))
            brush = tk.Color(*rng.uniform(0, 1, 3), float(rng.choice([1.0, 0.5])))
            if rng.uniform() < 0.2:
                brush = tk.LinearGradient((0, 0), (70, 50), [(0.0, brush), (1.0, tk.Color(0, 1, 0, 0.7))])
            canvas.push_path(path.close_path(), brush, rule=tk.FillRule(int(rng.integers(0, 2))))

    for k in range(depth):
        draw()
        canvas.push_clip_sdf_rect_layer(0.3 * k, 0.2 * k, 70 - 0.4 * k, 50 - 0.3 * k, 4.0)
    draw()
    for k in range(depth):
        canvas.pop_layer()
        draw()
    gpu, ref, bad = compare_frame(ctx, canvas)
    assert not bad, bad
