// What the one-kernel scan (pathscan.hip) costs a path beyond its share, which decides
// whether a frame takes it: at an upload by the host and tk_k_path_scan_check, else by
// the front end.  `visits` is the path's segment capacity, the tiles its lines visit.
#pragma once

#include "scan_line.h"

namespace tk {

// How far a path's lines go, as visits: what the separate stages take for its longest
// line, since they give a line a thread (and at most the path's box).
TK_HD inline uint32_t path_scan_reach(uint32_t lines, uint32_t visits, uint32_t tiles) {
    const uint64_t across = 3ull * tiles, along = 1024ull * visits / (lines ? lines : 1u);
    const uint64_t reach = across < along ? across : along;
    return reach < 0xFFFFFFFFull ? uint32_t(reach) : 0xFFFFFFFFu;
}

// A workgroup takes all of a path's lines and walks a line's tiles one after another, so
// the path takes some 5 ns a line and 3-9 ns a visit (the more, the fewer tiles the
// visits fall on).  In the stages only the longest line counts.  How far a path is past
// the point where they are as fast, in visits.
// Scan and coarse of one path, us, in one kernel and by the stages: 8,000 lines of about a
// visit each on 128x128, 512x512 and 4096x4096 119 and 105, 119 and 119, 282 and 314; 1,000
// lines across 128x128 (5.5 visits each), 512x512 (21), 1024x1024 (43) and 4096x4096
// (170) 117 and 122, 286 and 175, 403 and 246, 717 and 794; 4,000 such lines 274 and 146,
// 714 and 181, 1357 and 255, 2189 and 868.
TK_HD inline uint32_t path_scan_excess(uint32_t lines, uint32_t visits, uint32_t tiles) {
    const uint64_t even = 4096ull + lines + path_scan_reach(lines, visits, tiles);
    const uint32_t long_from = 6144u + (tiles < 1024u ? 2u * tiles : 2048u);
    const uint32_t over = visits > even ? visits - uint32_t(even) : 0u, longer = lines > long_from ? lines - long_from : 0u;
    return over > longer ? over : longer;
}

// A path of more tiles than two runs is shared by several workgroups, each of which takes
// all its lines: those workgroups, by their lines and visits over a fixed part.
constexpr uint32_t kPathScanSharedTiles = 1280u;
TK_HD inline uint64_t path_scan_shared(uint32_t lines, uint32_t visits, uint32_t tiles) {
    return tiles > kPathScanSharedTiles ? uint64_t(tiles / (kPathScanSharedTiles / 2u)) * (8192ull + lines + visits) : 0ull;
}

// Whether the one-kernel scan is the faster for a frame of `lines` lines, by its paths'
// largest excess, the largest reach of a shared one and the sum of the shared parts.  What
// it gains on every line, some 40 ps (50,000 paths of 11.3 M lines: 0.32 ms against 0.80),
// may pay for a long path in a large frame and for shared ones; and where one path reaches
// far, the stages take as long whatever the others do (a third of it, as a visit takes up
// to three times as long on few tiles).  Paths over all of 4096x4096, scan and coarse, us,
// in one kernel and by the stages: 64 of 4,000 and 8,000 lines 694 and 873, 873 and 774; 100
// of 1,000, 4,000 and 8,000 789 and 892, 967 and 902, 1252 and 807; 8 of 1,000 lines across
// it 1048 and 884; 100 strokes of 20 lines, one in a box so small that it is past its own
// point, 540 and 908; beside 200,000 paths of 24 lines, one of 16,384 lines 533 and 570, one
// of 60,000 858 and 719, 100 of 8,000 1474 and 1286; beside 1,000,000, one of 60,000 lines
// 2079 and 2437, 100 of 8,000 2666 and 2985, one of 4,000 across 4451 and 2876.
TK_HD inline uint64_t path_scan_most_excess(uint64_t lines, uint64_t reach) { return lines / 256u + reach / 3u; }
TK_HD inline bool path_scan_pays(uint64_t lines, uint64_t excess, uint64_t reach, uint64_t shared) {
    return excess <= path_scan_most_excess(lines, reach) && shared <= (1ull << 27) + 12u * lines;
}

}  // namespace tk
