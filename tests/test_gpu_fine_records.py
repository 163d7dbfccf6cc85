"""Records that fine takes as they stand in a tile's streams, by the stage entry: tags
it does not know draw nothing in an interpreted stream, and are colours in a stream of
colours (fine/interpreter.hlsli:21-219, specialized.hlsli:19-35)."""
import ctypes as C

import numpy as np
import pytest

from tileink_amd import _abi
from tileink_amd._abi import check, lib

pytestmark = pytest.mark.gpu

END, FILL, COLOR, END_CLIP = 0, 1, 2, 4
INTERPRETER, COLORS, SDF, MIXED = 0, 2, 3, 4
WHITE = 0xFFFFFFFF


def _fine(ctx, kinds, streams, batches=1):
    """One tile per stream of (tag, backdrop, rule, segment start, end, colour) records;
    of several batches the streams of batch 0 first."""
    ptcl, ranges = [], []
    for stream in streams:
        ranges.append((len(ptcl), len(ptcl) + len(stream)))
        ptcl += stream
    T = len(streams) // batches
    record = np.zeros(2, np.dtype(_abi.DrawRecord))
    record["sdf_offset"] = record["sdf_shadow_offset"] = _abi.INVALID
    paint = np.zeros(16, np.uint32)
    paint[0], paint[4] = _abi.BRUSH_SOLID, WHITE
    cfg = _abi.FineConfig(16 * T, 16, 0, T, T, 1, batches, 0, 16, 0, 0, 2, len(ptcl), 1)
    keep = [ctx.to_device(a) for a in (record.view(np.uint32), paint, np.zeros((1, 5), np.float32),
                                       np.array(ranges, np.uint32), np.array(kinds, np.uint32),
                                       np.array(ptcl, np.int64).astype(np.uint32))]
    inputs = _abi.FineInputs()
    (inputs.draws, inputs.paint, inputs.segments, inputs.tile_ptcl_ranges, inputs.tile_kinds,
     inputs.ptcl) = (b.ptr for b in keep)
    rgba = ctx.to_device(np.zeros(256 * T, np.uint32))
    check(lib().tk_fine(ctx.handle, C.byref(cfg), C.byref(inputs), rgba.ptr))
    ctx.synchronize()
    return rgba.read(np.uint32).reshape(16, T, 16).transpose(1, 0, 2).reshape(T, 256)


def test_unknown_tags_draw_nothing_or_a_colour(ctx):
    # beside the tags 14 and 255: each known tag and 256, 2^31 or so more
    tags = [14, 255] + [k + more for k in range(16) for more in (256, 1 << 15, (1 << 32) - 256)]
    red = 0xFF0000FF
    kinds, streams, want = [], [], []
    for tag in tags:
        kinds += [INTERPRETER, COLORS]
        streams.append([(FILL, 1, 0, 0, 0, 0), (tag, 1, 0, 0, 0, 0), (END, 0, 0, 0, 0, 0)])
        streams.append([(tag, 0, 0, 0, 0, red), (END, 0, 0, 0, 0, 0)])
        want += [WHITE, red]
        # the record after it is drawn all the same
        kinds.append(INTERPRETER)
        streams.append([(tag, 1, 0, 0, 0, 0), (COLOR, 0, 0, 0, 0, red), (END, 0, 0, 0, 0, 0)])
        want.append(red)
        # alone: nothing
        kinds.append(INTERPRETER)
        streams.append([(tag, 1, 0, 0, 0, 0), (END, 0, 0, 0, 0, 0)])
        want.append(0)
    got = _fine(ctx, kinds, streams)
    bad = np.nonzero((got != np.array(want, np.uint32)[:, None]).any(1))[0]
    assert bad.size == 0, [(hex(tags[b // 4]), b % 4, hex(got[b][0])) for b in bad[:6]]


def _over(pixel, color):
    """A colour over a pixel in FP32, as the blend rounds (shared/pixel.hlsli:7-66)."""
    scale = np.float32(1.0) / np.float32(255.0)
    src = np.array([(color >> s) & 255 for s in (0, 8, 16, 24)], np.float32) * scale
    if color >> 24 == 255:
        return src
    return pixel if color >> 24 == 0 else src + pixel * (np.float32(1.0) - src[3])


# records of one stream, and streams of many batches, around the walk's window of 64
@pytest.mark.parametrize("records,batches", [(1, 1), (2, 1), (63, 1), (64, 1), (65, 1), (200, 1), (1, 2), (3, 63), (2, 64),
                                             (1, 65), (5, 130)])
def test_colours_over_a_tile(ctx, records, batches):
    rng = np.random.default_rng(records + 1000 * batches)
    tiles = [COLORS, SDF, MIXED, INTERPRETER, COLORS]
    kinds, streams = [], []
    want = np.zeros((len(tiles), 4), np.float32)
    for b in range(batches):
        for t, kind in enumerate(tiles):
            # premultiplied, opaque and translucent, and some that draw nothing
            alpha = rng.choice([0, 1, 40, 128, 254, 255], records, p=[0.1, 0.1, 0.3, 0.2, 0.2, 0.1])
            stream = []
            for a in alpha:
                rgb = rng.integers(0, int(a) + 1, 3)
                color = int(rgb[0] | rgb[1] << 8 | rgb[2] << 16 | int(a) << 24)
                # a stream of colours takes any tag as one
                stream.append((FILL if kind == COLORS and t == 4 else COLOR, 3, 1, 0, 0, color))
                want[t] = _over(want[t], color)
            kinds.append(kind)
            streams.append(stream + [(END, 0, 0, 0, 0, 0), (COLOR, 0, 0, 0, 0, WHITE)])
            # the store between batches
            want[t] = np.trunc(np.clip(want[t] * np.float32(255) + np.float32(0.5), 0, 255)) * (np.float32(1) / np.float32(255))
    bytes_ = np.trunc(want * np.float32(255) + np.float32(0.5)).astype(np.uint32)
    expect = bytes_[:, 0] | bytes_[:, 1] << 8 | bytes_[:, 2] << 16 | bytes_[:, 3] << 24
    got = _fine(ctx, kinds, streams, batches)
    # In an interpreted stream a colour is scaled by its mask, 255 / 65025 rounded, not 1 / 255.
    plain = [t for t in range(len(tiles)) if tiles[t] != INTERPRETER]
    assert np.array_equal(got[plain], np.repeat(expect[plain, None], 256, 1))
    diff = np.abs(got[3, :, None].view(np.uint8).astype(int) - np.repeat(expect[3:4], 256)[:, None].view(np.uint8).astype(int))
    assert diff.max() <= 1
