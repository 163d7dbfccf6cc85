// The scan of a frame whose lines and backdrop slabs lie path by path, in one
// kernel; included by kernels.hip.
//
// The separate stages (scan_clear, scan_count, scan_prefix, cumsum, scan_emit)
// exchange their (path, tile) tables through memory, because each dispatch sees the
// lines of all paths.  But a path's counts, offsets, backdrop rows and segment slots
// depend on its own lines only (scan/count.hlsl:13-40, prefix_chunks.hlsl:16-38,
// cumsum.hlsl:16-71, emit.hlsl:14-28), and a recorder lays the paths out one after
// another.  So a workgroup takes a run of consecutive paths and carries it through:
// it counts into LDS, scans there, writes each table once, and emits the segments
// with LDS cursors.  Memory sees the lines twice, the tables once (no clear before,
// no atomics on them) and the segments.
//
// Run r covers the positions [r, r + 1) * RUN of the paths laid end to end, each as
// long as its lines, its tiles and four: it takes the paths that start there (a
// quarter of RUN at most), the last of which may reach beyond.  So the paths
// before the last hold fewer than one RUN of tiles, and a path of up to two more is
// counted in the same tables, three RUNs long.  A larger path leaves runs behind it in
// which no path starts; these share its tile rows out among them.  Each reads all the
// path's lines, tables its own rows, and finds where its segments start by counting
// the visits above them, so no workgroup waits on another.
//
// Most lines of flattened curves stay in one tile and need neither the traversal's
// quotients nor the clipping's, so each wave handles those as they come and queues
// the others, to take them 64 at a time.  A line's loads stand one step ahead, and
// its path comes from LDS: by the records, a step was a chain of three loads.
// Bound by VALU issue (45.5 M lines: 1.10 of 1.20 ms at four cycles an instruction) and,
// below a thousand runs, by the chain of loads from a run's search to its segments.  11.3 M lines of 50,000 paths, 2.3 M
// tiles, 14.8 M segments: 0.32 ms (the separate stages 0.80 ms, 0.45 ms of it beside
// coarse); 27 lines of an icon: 14 us (six launches before, 36 us with their gaps).

namespace {

// What a workgroup carries: paths [first, end), their lines, and the tiles
// [tile0, tile0 + tiles) of their slabs.
struct PathRun {
    uint32_t first, end, line0, line1, tile0, tiles;
    bool band;  // some tile rows of one path
};

__device__ __forceinline__ uint64_t path_scan_position(const tk_args_path_scan &a, uint32_t p) {
    return (uint64_t)a.paths[p].line_start + a.paths[p].data_offset + 4ull * p;
}

// Run r; false when nothing is left to it.  Its paths are found by a search, 64 probes
// a step (three steps for 262,144 paths), which the loads of one wave overlap: a
// table of them would be one more kernel and buffer in front of every scene.
__device__ __forceinline__ bool path_run(const tk_args_path_scan &a, uint32_t r, PathRun &u) {
    const Const<tk_path_record> paths = constant(a.paths);
    const uint64_t begin = (uint64_t)r * a.run, end = begin + a.run;
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lo = 0u, hi = a.path_count;  // the first path at or past `begin` is in [lo, hi]
    while (lo < hi) {
        const uint32_t step = (hi - lo + 63u) / 64u, probe = lo + lane * step;
        const uint32_t n = (uint32_t)__popcll(__ballot(probe < hi && path_scan_position(a, probe) < begin));
        hi = min(lo + n * step, hi);
        lo = n ? lo + (n - 1u) * step + 1u : lo;
    }
    u.first = u.end = uniform(lo);
    for (uint32_t n = 64u; n == 64u; u.end += n) {
        const uint32_t probe = u.end + lane;
        n = (uint32_t)__popcll(__ballot(probe < a.path_count && path_scan_position(a, probe) < end));
    }
    u.band = u.first >= u.end;
    if (!u.band) {
        if (paths[u.end - 1u].data_len > 2u * a.run) u.end -= 1u;  // the runs after this one
        if (u.first >= u.end) return false;
        const __attribute__((address_space(4))) tk_path_record &p = paths[u.first], &q = paths[u.end - 1u];
        u.line0 = p.line_start;
        u.line1 = q.line_start + q.line_count;
        u.tile0 = p.data_offset;
        u.tiles = q.data_offset + q.data_len - p.data_offset;
        return u.tiles <= 3u * a.run;
    }
    if (u.first == 0u) return false;
    u.end = u.first;
    u.first -= 1u;
    const __attribute__((address_space(4))) tk_path_record &p = paths[u.first];
    if (p.data_len <= 2u * a.run) return false;
    const uint64_t at = (uint64_t)p.line_start + p.data_offset + 4ull * u.first;
    const uint32_t k0 = (uint32_t)(at / a.run);
    const uint32_t k1 = (uint32_t)((at + p.line_count + p.data_len + 4u) / a.run);
    const uint32_t bands = k1 - k0 - 1u, rows = p.tile_y1 - p.tile_y0, width = p.tile_x1 - p.tile_x0;
    const uint32_t share = (rows + bands - 1u) / bands, row = (r - k0 - 1u) * share;
    if (row >= rows) return false;
    u.line0 = p.line_start;
    u.line1 = p.line_start + p.line_count;
    u.tile0 = p.data_offset + row * width;
    u.tiles = min(share, rows - row) * width;
    return u.tiles <= 3u * a.run;
}

// What a run keeps of each of its paths in LDS: its first tile less the run's, its
// box {x0 | y0 << 16, x1 | flags | y1 << 16}, and its segments' start less the slots
// before it in the run (once those are known).
constexpr uint32_t kPathIdentity = 1u << 15, kPathLeftOut = 1u << 14;
struct alignas(16) RunPath {
    uint32_t first, low, high, offset;
};
static_assert(TK_PATH_SCAN_RUN < kPathLeftOut, "x1 and the flags share 16 bits");

__device__ __forceinline__ bool is_identity(const tk_affine &t) {
    return t.a == 1.0f && t.b == 0.0f && t.c == 0.0f && t.d == 1.0f && t.e == 0.0f && t.f == 0.0f;
}

// A line's box and end points; false when an incremental render leaves its path out
// or the box is empty.  data_offset is relative to the run.
__device__ __forceinline__ bool path_scan_line(const tk_args_path_scan &a, const tk_line &line, const RunPath &p,
                                               ScanTraversal &s) {
    s = ScanTraversal{};
    s.data_offset = p.first;
    s.bx = p.low & 0xFFFFu;
    s.by = p.low >> 16;
    s.bz = p.high & (kPathLeftOut - 1u);
    s.bw = p.high >> 16;
    if ((p.high & kPathLeftOut) || s.bx >= s.bz || s.by >= s.bw) return false;
    tk_affine t{1.0f, 0.0f, 0.0f, 1.0f, 0.0f, 0.0f};
    if (!(p.high & kPathIdentity)) t = a.paths[line.path_id].transform;
    scan_endpoints(line, t, s);
    return true;
}

// Passes the workgroup's lines: one(s, path, tx, ty) for a line in one tile, many(s,
// path) for any other that visits tiles; `path` is its RunPath.  `queue`: the wave's,
// 128 entries.
template <class One, class Many>
__device__ __forceinline__ void path_scan_lines(const tk_args_path_scan &a, const PathRun &u, const RunPath *paths,
                                                uint16_t *queue, One one, Many many) {
    const uint32_t lane = threadIdx.x & 63u, n = u.line1 - u.line0;
    const auto load = [&](uint32_t index) { return index < n ? a.lines[u.line0 + index] : tk_line{}; };
    const auto order = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    const auto general = [&](uint32_t index) {
        const tk_line line = load(index);
        const RunPath path = paths[line.path_id - u.first];
        ScanTraversal s;
        if (path_scan_line(a, line, path, s) && scan_traverse(s)) many(s, path);
    };
    uint32_t held = 0u;  // fewer than 64 queued between steps
    const uint32_t wave_base = uniform(threadIdx.x & ~63u);
    tk_line next = load(wave_base + lane);
    for (uint32_t base = wave_base; base < n; base += 256u) {
        const uint32_t index = base + lane;
        const tk_line line = next;
        next = load(index + 256u);
        bool queued = false;
        if (index < n) {
            const RunPath path = paths[line.path_id - u.first];
            ScanTraversal s;
            if (path_scan_line(a, line, path, s)) {
                int32_t tx, ty;
                const ScanSingle single = scan_single_tile(s, tx, ty);
                if (single == kScanOne) one(s, path, tx, ty);
                queued = single == kScanGeneral;
            }
        }
        const uint64_t mask = __ballot(queued);
        if (queued) queue[held + (uint32_t)__popcll(mask & lanes_below(lane))] = (uint16_t)index;
        held += (uint32_t)__popcll(mask);
        order();
        if (held >= 64u) {
            held -= 64u;
            general(queue[held + lane]);
            order();
        }
    }
    if (lane < held) general(queue[lane]);
    order();
}

}  // namespace

extern "C" __global__ __launch_bounds__(256) void tk_k_path_scan(tk_args_path_scan a) {
    // Its paths, at most RUN / 4; per tile the visits, then the slots before it among
    // the run's (one word past the end for the last's); per tile the backdrop delta,
    // then the deltas' running sum.
    extern __shared__ uint32_t path_scan_lds[];  // TK_PATH_SCAN_LDS(run)
    RunPath *paths = reinterpret_cast<RunPath *>(path_scan_lds);
    uint32_t *slots = path_scan_lds + 4u * ((a.run + 3u) / 4u), *deltas = slots + 3u * a.run + 1u;
    __shared__ uint16_t queues[4][128];
    __shared__ uint32_t sums[2][2][4], s_before;
    static_assert(TK_PATH_SCAN_LINES + TK_PATH_SCAN_RUN < 65536u, "the queues hold line numbers in 16 bits");
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = uniform(tid >> 6);
#pragma unroll
    for (uint32_t k = 0; k < 5u; ++k)  // tables that later kernels of the frame start from
        for (uint64_t i = blockIdx.x * 256ull + tid; i < a.clear[k].count; i += gridDim.x * 256ull)
            a.clear[k].words[i] = a.clear[k].value;
    if (blockIdx.x >= a.runs) {  // the workgroups behind the runs build the draw tables, a launch less
        draw_tables(a.tables, (blockIdx.x - a.runs) * 256u + tid);
        return;
    }
    PathRun u;
    if (!path_run(a, blockIdx.x, u)) return;
    const uint32_t path_count = u.end - u.first;  // at most RUN / 4
    uint32_t path_end = 0u;                       // thread j: path j's tiles end here
    bool last_part = true;                        // and with them the path
    if (tid < path_count) {
        const tk_path_record &p = a.paths[u.first + tid];
        const bool left_out = a.path_active && a.path_active[u.first + tid] == 0u;
        paths[tid] = RunPath{p.data_offset - u.tile0, p.tile_x0 | (p.tile_y0 << 16),
                             p.tile_x1 | (is_identity(p.transform) ? kPathIdentity : 0u) |
                                 (left_out ? kPathLeftOut : 0u) | (p.tile_y1 << 16),
                             p.segment_start};
        path_end = p.data_offset - u.tile0 + p.data_len;
        last_part = path_end <= u.tiles;
        path_end = min(path_end, u.tiles);
    }
    for (uint32_t t = tid; t < u.tiles; t += 256u) {
        slots[t] = 0u;
        deltas[t] = 0u;
    }
    if (tid == 0u) s_before = 0u;
    __syncthreads();

    uint32_t before = 0u;  // visits above a band
    path_scan_lines(
        a, u, paths, queues[wave],
        [&](const ScanTraversal &s, const RunPath &, int32_t tx, int32_t ty) {
            const uint32_t t = scan_tile_offset(s, tx, ty);
            if (t < u.tiles) {
                const bool top = fabsf((float)ty - s.py0 * (1.0f / 16.0f)) <= kScanEpsilon;
                if (top && tx + 1 < (int32_t)s.bz) atomicAdd(&deltas[t + 1u], s.down ? ~0u : 1u);
                atomicAdd(&slots[t], 1u);
            } else if ((int32_t)t < 0) {
                ++before;
            }
        },
        [&](const ScanTraversal &s, const RunPath &) {
            const uint32_t step = s.down ? ~0u : 1u, stride = s.bz - s.bx;
            for (int32_t y = s.ymin; y < s.ymax; y++) {
                const uint32_t t = s.data_offset + (uint32_t)(y - (int32_t)s.by) * stride;
                if (t < u.tiles) atomicAdd(&deltas[t], step);
            }
            float last_z = floorf(s.a * ((float)s.imin - 1.0f) + s.b);
            for (uint32_t i = s.imin; i < s.imax; i++) {
                const float z = floorf(s.a * (float)i + s.b);
                int32_t tx, ty;
                scan_tile(s, i, z, tx, ty);
                if (scan_tile_inside(s, tx, ty)) {
                    const uint32_t t = scan_tile_offset(s, tx, ty);
                    if (t < u.tiles) {
                        bool top = last_z == z;
                        if (i == 0u) top = fabsf(s.y0 - s.py0 * (1.0f / 16.0f)) <= kScanEpsilon;
                        // the tile to the right is of the same row, so of the same band
                        if (top && tx + 1 < (int32_t)s.bz) atomicAdd(&deltas[t + 1u], step);
                        atomicAdd(&slots[t], 1u);
                    } else if ((int32_t)t < 0) {
                        ++before;
                    }
                }
                last_z = z;
            }
        });
    if (u.band) {
        before = wave_sum_u32(before);
        if (lane == 0u && before) atomicAdd(&s_before, before);
    }
    __syncthreads();

    // Both tables' prefix sums over the whole run; what belongs to one path or row
    // alone is a difference of two of them.
    uint32_t slot_carry = 0u, delta_carry = 0u;
    for (uint32_t base = 0u, buffer = 0u; base < u.tiles; base += 256u, buffer ^= 1u) {
        const uint32_t t = base + tid;
        const uint32_t v = t < u.tiles ? slots[t] : 0u, d = t < u.tiles ? deltas[t] : 0u;
        const uint32_t vi = wave_inclusive_scan_dpp(v), di = wave_inclusive_scan_dpp(d);
        if (lane == 63u) {
            sums[buffer][0][wave] = vi;
            sums[buffer][1][wave] = di;
        }
        __syncthreads();
        uint32_t v_before = slot_carry, d_before = delta_carry;
#pragma unroll
        for (uint32_t w = 0; w < 4u; ++w) {
            const uint32_t vs = sums[buffer][0][w], ds = sums[buffer][1][w];
            if (w < wave) v_before += vs, d_before += ds;
            slot_carry += vs;
            delta_carry += ds;
        }
        if (t < u.tiles) {
            slots[t] = v_before + vi - v;
            deltas[t] = d_before + di;
        }
    }
    if (tid == 0u) slots[u.tiles] = slot_carry;
    __syncthreads();
    if (tid < path_count) {
        const uint32_t first = u.band ? 0u : slots[paths[tid].first], above = u.band ? s_before : 0u;
        if (last_part) a.bumps[u.first + tid] = slots[path_end] - first + above;
        paths[tid].offset += above - first;
    }
    __syncthreads();
    for (uint32_t t = tid; t < u.tiles; t += 256u) {
        uint32_t lo = 0u, hi = path_count;  // the last path whose first tile is at or before t
        while (hi - lo > 1u) {
            const uint32_t mid = (lo + hi) >> 1;
            if (paths[mid].first <= t) lo = mid;
            else hi = mid;
        }
        const RunPath p = paths[lo];
        const uint32_t first = u.band ? 0u : p.first, stride = (p.high & (kPathLeftOut - 1u)) - (p.low & 0xFFFFu);
        const uint32_t start = p.offset + slots[t], end = p.offset + slots[t + 1u];
        // exact: below 2^12 over at most 2^10, half a step from the nearest whole number
        const uint32_t row = first + (uint32_t)(((float)(t - first) + 0.5f) * (1.0f / (float)stride)) * stride;
        const uint32_t tile = u.tile0 + t;
        a.counts[tile] = end - start;
        a.ranges[tile] = tk_segment_range{start, end};
        a.cursors[tile] = end;  // as emission leaves it
        if (a.raw_backdrops) a.raw_backdrops[tile] = (int32_t)(deltas[t] - (t ? deltas[t - 1u] : 0u));
        a.backdrops[tile] = (int32_t)(deltas[t] - (row ? deltas[row - 1u] : 0u));
    }
    __syncthreads();

    path_scan_lines(
        a, u, paths, queues[wave],
        [&](const ScanTraversal &s, const RunPath &path, int32_t tx, int32_t ty) {
            const uint32_t t = scan_tile_offset(s, tx, ty);
            if (t >= u.tiles) return;
            const uint32_t slot = path.offset + atomicAdd(&slots[t], 1u);
            if (slot < a.cfg.segment_capacity)
                a.segments[slot] = tile_segment(s.px0, s.py0, s.px1, s.py1, (float)tx * kTileSize, (float)ty * kTileSize, s.down);
        },
        [&](const ScanTraversal &s, const RunPath &path) {
            for (uint32_t i = s.imin; i < s.imax; i++) {
                const float z = floorf(s.a * (float)i + s.b);
                int32_t tx, ty;
                scan_tile(s, i, z, tx, ty);
                if (!scan_tile_inside(s, tx, ty)) continue;
                const uint32_t t = scan_tile_offset(s, tx, ty);
                if (t >= u.tiles) continue;
                const uint32_t slot = path.offset + atomicAdd(&slots[t], 1u);
                if (slot < a.cfg.segment_capacity) a.segments[slot] = clipped_segment(s, i, z, tx, ty);
            }
        });
}

// Whether a scene is laid out as tk_k_path_scan takes it: lines and slabs path by
// path without gaps, slabs as large as their tile boxes, scan chunks and cumsum rows
// that cut every slab as the recorder does, no path of more than TK_PATH_SCAN_LINES
// lines or too long for the frame (path_scan_rule.h), and no box beyond the canvas or, where that is wider, beyond TK_PATH_SCAN_RUN.
// Anything else is left to the separate stages, whose result for it is the
// reference's.  One thread per line, path, chunk and row; 5 us of an upload of 3,900
// lines (75 -> 80 us), 9 of one of 107,000 (216 -> 237), 198 of one of 45.5 M.
extern "C" __global__ __launch_bounds__(256) void tk_k_path_scan_check(tk_args_path_scan_check a) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const tk_scan_config &cfg = a.cfg;
    bool ok = true;
    if (i < cfg.path_count) {
        const tk_path_record &p = a.paths[i];
        const bool last = i + 1u == cfg.path_count;
        ok = p.line_start == (i ? a.paths[i - 1u].line_start + a.paths[i - 1u].line_count : 0u) &&
             p.data_offset == (i ? a.paths[i - 1u].data_offset + a.paths[i - 1u].data_len : 0u) &&
             p.line_count <= cfg.line_count - min(p.line_start, cfg.line_count) &&
             p.data_len <= cfg.backdrop_len - min(p.data_offset, cfg.backdrop_len) &&
             (!last || (p.line_start + p.line_count == cfg.line_count && p.data_offset + p.data_len == cfg.backdrop_len)) &&
             p.tile_x0 <= p.tile_x1 && p.tile_y0 <= p.tile_y1 && p.tile_x1 <= a.widest && p.tile_y1 <= 0xFFFFu &&
             (uint64_t)(p.tile_x1 - p.tile_x0) * (p.tile_y1 - p.tile_y0) == p.data_len &&
             p.line_count <= TK_PATH_SCAN_LINES &&
             tk::path_scan_excess(p.line_count, p.segment_capacity, p.data_len) <= a.most_excess;
        const tk_scan_chunk_range r = a.chunk_ranges[i];
        ok = ok && r.start == (i ? a.chunk_ranges[i - 1u].end : 0u) && r.end >= r.start &&
             r.end - r.start == (p.data_len + TK_SCAN_CHUNK_SIZE - 1u) / TK_SCAN_CHUNK_SIZE &&
             (!last || r.end == cfg.scan_chunk_count);
    }
    if (i < cfg.line_count) {
        const uint32_t p = a.lines[i].path_id;
        ok = ok && p < cfg.path_count && i - a.paths[p].line_start < a.paths[p].line_count;
    }
    if (i < cfg.scan_chunk_count) {
        const tk_scan_chunk c = a.chunks[i];
        if (c.path_id < cfg.path_count) {
            const tk_path_record &p = a.paths[c.path_id];
            const tk_scan_chunk_range r = a.chunk_ranges[c.path_id];
            const uint32_t at = (i - r.start) * TK_SCAN_CHUNK_SIZE;
            ok = ok && i >= r.start && i < r.end && at < p.data_len && c.backdrop_offset == p.data_offset + at &&
                 c.len == min((uint32_t)TK_SCAN_CHUNK_SIZE, p.data_len - at);
        } else {
            ok = false;
        }
    }
    if (i < a.row_count) {
        // The row's tiles [at, end), from chunks that follow each other and each other's rows.
        const uint32_t c0 = a.row_starts[i], c1 = a.row_ends[i];
        bool row_ok = c0 < c1 && c1 <= a.cs_chunk_count && (i ? c0 != 0u && a.row_ends[i - 1u] == c0 : c0 == 0u) &&
                      (i + 1u < a.row_count || c1 == a.cs_chunk_count) && c1 - c0 <= TK_PATH_SCAN_RUN;
        if (row_ok) {
            const uint32_t at = a.cs_offsets[c0];
            uint32_t end = at;
            for (uint32_t c = c0; c < c1; ++c) {
                row_ok = row_ok && a.cs_offsets[c] == end && a.cs_lens[c] >= 1u && a.cs_lens[c] <= TK_CUMSUM_CHUNK_SIZE;
                end += min(a.cs_lens[c], (uint32_t)TK_CUMSUM_CHUNK_SIZE);
            }
            const uint32_t expect = i ? a.cs_offsets[c0 - 1u] + a.cs_lens[c0 - 1u] : 0u;
            row_ok = row_ok && at == expect && (i + 1u < a.row_count || end == cfg.backdrop_len);
            // the last path whose slab starts at or before the row, empty ones passed over
            uint32_t lo = 0u, hi = cfg.path_count;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (a.paths[mid].data_offset <= at) lo = mid + 1u;
                else hi = mid;
            }
            row_ok = row_ok && lo != 0u;
            if (row_ok) {
                const tk_path_record &p = a.paths[lo - 1u];
                const uint32_t width = p.tile_x1 - p.tile_x0;
                row_ok = width != 0u && at - p.data_offset < p.data_len && (at - p.data_offset) % width == 0u &&
                         end - at == width;
            }
        }
        ok = ok && row_ok;
    }
    if (i == 0u && ((cfg.path_count == 0u && (cfg.line_count || cfg.backdrop_len)) || (a.row_count == 0u && cfg.backdrop_len)))
        ok = false;
    if (!ok) *a.refused = 1u;
}
