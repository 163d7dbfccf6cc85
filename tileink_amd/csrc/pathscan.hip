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
// Run r covers the positions [r, r + 1) * TK_PATH_SCAN_RUN of the line and tile
// counts summed over the paths: it takes the paths that start there, the last of
// which may reach beyond.  So the paths before the last hold fewer than one RUN of
// tiles, and a path of up to two more is counted in the same tables, three RUNs
// long.  A larger path leaves runs behind it in which no path starts; these share its
// tile rows out among them.  Each reads all the path's lines, tables its own rows,
// and finds where its segments start by counting the visits above them, so no
// workgroup waits on another.

namespace {

constexpr uint32_t kPathScanTiles = 3u * TK_PATH_SCAN_RUN;

// What a workgroup carries: paths [first, end), their lines, and the tiles
// [tile0, tile0 + tiles) of their slabs.
struct PathRun {
    uint32_t first, end, line0, line1, tile0, tiles;
    bool band;  // some tile rows of one path
};

__device__ __forceinline__ uint64_t path_scan_position(const tk_args_path_scan &a, uint32_t p) {
    return (uint64_t)a.paths[p].line_start + a.paths[p].data_offset;
}

// Run r; false when nothing is left to it.  Its paths are found by a search, 64 probes
// a step (three steps for 262,144 paths), which the loads of one wave overlap: a
// table of them would be one more kernel and buffer in front of every scene.
__device__ __forceinline__ bool path_run(const tk_args_path_scan &a, uint32_t r, PathRun &u) {
    const Const<tk_path_record> paths = constant(a.paths);
    const uint64_t begin = (uint64_t)r * TK_PATH_SCAN_RUN, end = begin + TK_PATH_SCAN_RUN;
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
        if (paths[u.end - 1u].data_len > 2u * TK_PATH_SCAN_RUN) u.end -= 1u;  // the runs after this one
        if (u.first >= u.end) return false;
        const __attribute__((address_space(4))) tk_path_record &p = paths[u.first], &q = paths[u.end - 1u];
        u.line0 = p.line_start;
        u.line1 = q.line_start + q.line_count;
        u.tile0 = p.data_offset;
        u.tiles = q.data_offset + q.data_len - p.data_offset;
        return u.tiles <= kPathScanTiles;
    }
    if (u.first == 0u) return false;
    u.end = u.first;
    u.first -= 1u;
    const __attribute__((address_space(4))) tk_path_record &p = paths[u.first];
    if (p.data_len <= 2u * TK_PATH_SCAN_RUN) return false;
    const uint32_t k0 = (uint32_t)(((uint64_t)p.line_start + p.data_offset) / TK_PATH_SCAN_RUN);
    const uint32_t k1 = (uint32_t)(((uint64_t)p.line_start + p.line_count + p.data_offset + p.data_len) / TK_PATH_SCAN_RUN);
    const uint32_t bands = k1 - k0 - 1u, rows = p.tile_y1 - p.tile_y0, width = p.tile_x1 - p.tile_x0;
    const uint32_t share = (rows + bands - 1u) / bands, row = (r - k0 - 1u) * share;
    if (row >= rows) return false;
    u.line0 = p.line_start;
    u.line1 = p.line_start + p.line_count;
    u.tile0 = p.data_offset + row * width;
    u.tiles = min(share, rows - row) * width;
    return u.tiles <= kPathScanTiles;
}

// The traversal of line `id`, unless an incremental render leaves its path out.
__device__ __forceinline__ bool path_scan_line(const tk_args_path_scan &a, uint32_t id, ScanTraversal &s) {
    if (a.path_active) {
        const uint32_t path = a.lines[id].path_id;
        if (path < a.path_count && a.path_active[path] == 0u) return false;
    }
    return scan_geometry(a.lines, a.paths, a.path_count, id, s);
}

}  // namespace

extern "C" __global__ __launch_bounds__(256) void tk_k_path_scan(tk_args_path_scan a) {
    __shared__ uint32_t counts[kPathScanTiles], deltas[kPathScanTiles];
    __shared__ uint32_t s_before;
#pragma unroll
    for (uint32_t k = 0; k < 3u; ++k)  // words that later kernels of the frame start from zero
        for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < a.clear[k].count; i += gridDim.x * 256ull)
            a.clear[k].words[i] = 0u;
    PathRun u;
    if (!path_run(a, blockIdx.x, u)) return;
    for (uint32_t t = threadIdx.x; t < u.tiles; t += 256u) {
        counts[t] = 0u;
        deltas[t] = 0u;
    }
    if (threadIdx.x == 0u) s_before = 0u;
    __syncthreads();

    uint32_t before = 0u;  // visits above a band
    for (uint32_t id = u.line0 + threadIdx.x; id < u.line1; id += 256u) {
        ScanTraversal s;
        if (!path_scan_line(a, id, s)) continue;
        const uint32_t step = s.down ? ~0u : 1u, stride = s.bz - s.bx, base = s.data_offset - u.tile0;
        for (int32_t y = s.ymin; y < s.ymax; y++) {
            const uint32_t t = base + (uint32_t)(y - (int32_t)s.by) * stride;
            if (t < u.tiles) atomicAdd(&deltas[t], step);
        }
        float last_z = floorf(s.a * ((float)s.imin - 1.0f) + s.b);
        for (uint32_t i = s.imin; i < s.imax; i++) {
            const float z = floorf(s.a * (float)i + s.b);
            int32_t tx, ty;
            scan_tile(s, i, z, tx, ty);
            if (scan_tile_inside(s, tx, ty)) {
                const uint32_t offset = scan_tile_offset(s, tx, ty), t = offset - u.tile0;
                if (t < u.tiles) {
                    bool top = last_z == z;
                    if (i == 0u) top = fabsf(s.y0 - s.py0 * (1.0f / 16.0f)) <= kScanEpsilon;
                    // the tile to the right is of the same row, so of the same band
                    if (top && tx + 1 < (int32_t)s.bz) atomicAdd(&deltas[t + 1u], step);
                    atomicAdd(&counts[t], 1u);
                } else if (offset < u.tile0) {
                    ++before;
                }
            }
            last_z = z;
        }
    }
    if (u.band) {
        before = wave_sum_u32(before);
        if (__lane_id() == 0u && before) atomicAdd(&s_before, before);
    }
    __syncthreads();

    // One wave per path, its tiles in order, 64 at a time: the slots before each tile
    // and the running sum of the deltas.
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t p = u.first + uniform(threadIdx.x >> 6); p < u.end; p += 4u) {
        const __attribute__((address_space(4))) tk_path_record &r = constant(a.paths)[p];
        const uint32_t first = u.band ? u.tile0 : r.data_offset, n = u.band ? u.tiles : r.data_len;
        const uint32_t o = first - u.tile0, stride = r.tile_x1 - r.tile_x0, start = r.segment_start;
        uint32_t slot = start + (u.band ? s_before : 0u), sum = 0u;
        for (uint32_t c = 0u; c < n; c += 64u) {
            const uint32_t i = c + lane;
            const uint32_t v = i < n ? counts[o + i] : 0u, d = i < n ? deltas[o + i] : 0u;
            const uint32_t end = slot + wave_inclusive_scan_dpp(v), total = sum + wave_inclusive_scan_dpp(d);
            if (i < n) {
                a.counts[first + i] = v;
                a.ranges[first + i] = tk_segment_range{end - v, end};
                a.cursors[first + i] = end;  // as emission leaves it
                if (a.raw_backdrops) a.raw_backdrops[first + i] = (int32_t)d;
                counts[o + i] = end - v;
                deltas[o + i] = total;
            }
            slot = (uint32_t)__builtin_amdgcn_readlane((int)end, 63);
            sum = (uint32_t)__builtin_amdgcn_readlane((int)total, 63);
        }
        if (lane == 0u && first + n == r.data_offset + r.data_len) a.bumps[p] = slot - start;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // A tile's backdrop: the sum up to it less the sum before its row.
        for (uint32_t i = lane; i < n; i += 64u) {
            const uint32_t row = i - i % stride;
            a.backdrops[first + i] = (int32_t)(deltas[o + i] - (row ? deltas[o + row - 1u] : 0u));
        }
    }
    __syncthreads();

    for (uint32_t id = u.line0 + threadIdx.x; id < u.line1; id += 256u) {
        ScanTraversal s;
        if (!path_scan_line(a, id, s)) continue;
        for (uint32_t i = s.imin; i < s.imax; i++) {
            const float z = floorf(s.a * (float)i + s.b);
            int32_t tx, ty;
            scan_tile(s, i, z, tx, ty);
            if (!scan_tile_inside(s, tx, ty)) continue;
            const uint32_t t = scan_tile_offset(s, tx, ty) - u.tile0;
            if (t >= u.tiles) continue;
            const uint32_t slot = atomicAdd(&counts[t], 1u);
            if (slot < a.cfg.segment_capacity) a.segments[slot] = clipped_segment(s, i, z, tx, ty);
        }
    }
}

// Whether a scene is laid out as tk_k_path_scan takes it: lines and slabs path by
// path without gaps, slabs as large as their tile boxes, scan chunks and cumsum rows
// that cut every slab as the recorder does, and no path too long or too wide.
// Anything else is left to the separate stages, whose result for it is the
// reference's.  One thread per line, path, chunk and row.
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
             p.tile_x0 <= p.tile_x1 && p.tile_y0 <= p.tile_y1 && p.tile_x1 - p.tile_x0 <= TK_PATH_SCAN_RUN &&
             (uint64_t)(p.tile_x1 - p.tile_x0) * (p.tile_y1 - p.tile_y0) == p.data_len &&
             p.line_count <= TK_PATH_SCAN_LINES;
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
