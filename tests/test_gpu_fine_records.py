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
INTERPRETER, COLORS = 0, 2
WHITE = 0xFFFFFFFF


def _fine(ctx, kinds, streams):
    """One tile per stream of (tag, backdrop, rule, segment start, end, colour) records."""
    ptcl, ranges = [], []
    for stream in streams:
        ranges.append((len(ptcl), len(ptcl) + len(stream)))
        ptcl += stream
    T = len(streams)
    record = np.zeros(2, np.dtype(_abi.DrawRecord))
    record["sdf_offset"] = record["sdf_shadow_offset"] = _abi.INVALID
    paint = np.zeros(16, np.uint32)
    paint[0], paint[4] = _abi.BRUSH_SOLID, WHITE
    cfg = _abi.FineConfig(16 * T, 16, 0, T, T, 1, 1, 0, 16, 0, 0, 2, len(ptcl), 1)
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
