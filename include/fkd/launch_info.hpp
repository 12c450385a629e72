// fkd/launch_info.hpp -- what a launcher reports about the launch it made, and the geometry it hands to the kernels:
// shared by the launchers of the ahead-of-time kernels, the launcher of the run-time compiled ones and the kernels
// themselves (plain C++, no HIP).
#pragma once

namespace fkd {

struct LaunchInfo {
    const char* kernel;   // "rows", "rows_unaligned" (chains with a kernel of its own for such rows), "gather", "strip" or "divergent"
    unsigned grid[3], block[3];
    unsigned lds_bytes;
    // The kernel by its own name, where `kernel` is the name of the form it took the place of: "rows", "flat" (planes without gaps), "tiles", "strip",
    // "strip_lines" (stores moved on to line boundaries) or "divergent".
    const char* form;
};

// ---- the geometry a launcher hands to kernels that renumber their workgroups ----

// A run-time compiled kernel takes a TileGeom whichever form its launch has.  A launch of the strip form of the bilinear
// kernel has no tiles: its TileGeom has tiles_x == 0 and carries in n_tiles what strip_first_late_workgroup() says about it.
// kStreamFlag in n_tiles: the output of the run-time compiled bilinear kernel is streamed past the last-level cache (the
// ahead-of-time kernels are told by their type).
// (Four words: with a fifth, launches of few waves took 0.15 us longer, 8 crops to 224x224 3.96 instead of 3.80 us each.)
// kAnyPitchFlag beside it: a launch of the strip form whose source rows do not share their alignment.
constexpr unsigned kStreamFlag = 0x80000000u, kAnyPitchFlag = 0x40000000u;
struct TileGeom {
    unsigned tiles_x, tiles_y, n_tiles;
    // floor(2^32 / tiles_x) + 1 when (t * magic) >> 32 == t / tiles_x for every tile number t of a plane, else 0: the
    // division then costs two scalar multiplications instead of a float reciprocal on the vector unit.
    unsigned tiles_x_magic;
};
// Planar outputs of the bilinear kernel above this many bytes are stored with the non-temporal hint.  Written through the
// L2 they are kept by the 256 MB last-level cache, which pushes the source images out of it; every tap line then comes from
// HBM between the writes, one isolated read at a time, and each costs the channel a turn from writing to reading and back.
// 64 crops of a 3840x2160 image to 640x640 (314 MB out, 25 MB of source): 77 us written through, 60 us non-temporal, although
// the stores alone take 55 us either way.
// The line lies where a program that fills three such outputs in turn crosses it: at a third of that cache.  64 crops of a 1280x853
// image, written through / non-temporal: 224x457 (75 MiB) 15.8 / 16.1 us, 224x512 (84) 19.3 / 16.9, 224x670 (110) 26.3 / 21.4; rows of no
// whole lines, whose partial lines cost more without the cache to gather them: 225x455 (75) 19.3 / 26.1, 225x509 (84) 30.2 / 28.2, 225x667
// (110) 50 / 38, 36x2503 (66) 25.8 / 35.6.
// What it costs: a program with one output buffer, which would have stayed in the cache up to twice that size, writes slower and finds
// its output in HBM.  One buffer, launch alone: 224x670 19.6 / 21.2, 225x667 23.8 / 38.5; with a reader of the output (a conversion to
// bfloat16) behind each launch: 224x670 49.4 / 50.8, 225x667 53.0 / 57.6, 500x436 (160) 71 / 80; from 190 MiB on even these gain (224x1401,
// 230 MiB 110 / 97).  Three buffers with a reader: 225x667 67 / 64, 500x518 (190) 123 / 106.
constexpr unsigned long long kStreamOutputBytes = 80ull << 20;
// Launches of the rows kernel that write no more than this store without the non-temporal hint: with it
// a launch is not over before its last lines have left the chip.  us per launch, with the hint / without: 4 uchar3 images of 225x165
// (0.4 MB) 2.32 / 2.01, of 943x179 (2.0 MB) 2.93 / 2.68, of 886x260 (2.8 MB) 3.21 / 2.97; 30 operations on 1544x90 floats (0.6 MB)
// 2.20 / 1.91; P010 to float3 at 404x862 (4.2 MB) 3.07 / 2.93; UYVY to float3 at 1552x284 (5.3 MB) 2.44 / 2.67; RGB to UYVY at 2460x714 (3.5
// MB) 3.80 / 3.56, at 3638x632 (4.6 MB) 4.09 / 4.32; 100 images of 75x200 (4.5 MB) 6.5 / 6.1, of 228x113 (7.7 MB) 4.4 / 4.8, of 361x467 (51 MB) 20.9 / 25.9.
constexpr unsigned long long kSmallOutputBytes = 4ull << 20;
// The magic for dividing numbers below `limit` by d, or 0 when there is none.
inline unsigned division_magic(unsigned d, unsigned limit) {
    if (d == 0) return 0;
    const unsigned long long m = (1ull << 32) / d + 1;        // m * d - 2^32 is in (0, d]; exact while n * d < 2^32
    return (m < (1ull << 32) && (unsigned long long)limit * d < (1ull << 32)) ? unsigned(m) : 0u;
}

// Rows kernel, bands form of grid: launches of kRowsBandBlocks blocks per plane or more are one-dimensional, 8 *
// rows_band_chunk(blocks) workgroups per plane (see rows_in_bands in the kernels' header).
inline constexpr unsigned rows_band_chunk(unsigned blocks) { return (blocks + 7u) / 8u; }
constexpr unsigned kRowsBandBlocks = 4096;

// Scattered reads (points_body in the kernels' header): smaller launches keep the two-dimensional grid, whose workgroups are renumbered
// into bands as well (TileGeom::n_tiles == 0).  us without / with: 3 launches in turn each, perspective 686x1247 (4 of them) 26.4 / 20.9, 4 of
// 811x319 (320 blocks) 13.7 / 12.1, 4 of 336x905 (454) 14.5 / 12.0.  Not with a few blocks, whose launches are over before a second
// XCD asks for the same line (4 of 141x351, 88 blocks 9.4 / 9.6), nor where one block spans the row (4 of 187x1511 11.6 / 11.75).
inline bool rows_bands_2d(unsigned gx, unsigned gy) {
    return gx >= 2u && (unsigned long long)gx * gy >= 256u && division_magic(gx, gx * gy) != 0u;
}

// Bits 8 to 15 of a chain's Params::reserved: by how many elements at most the rows kernel's waves begin left of a row so
// that they store whole lines (Chain::finalize_write); the grid has to reach that much further.
inline constexpr unsigned rows_phase_bound(unsigned reserved) { return (reserved >> 8) & 0xffu; }

// Strip form of the bilinear kernel: a launch of at most kStripOneRoundWorkgroups workgroups (eight per compute unit: every
// workgroup resident from the start) runs with wave priorities; the kernel is told the number of the first workgroup that
// counts as started late, or 0 for a launch whose waves keep the default priority (see the kernels' header).
constexpr unsigned kStripOneRoundWorkgroups = 2048, kComputeUnits = 256, kStripLateWorkgroup = 4;
inline unsigned strip_first_late_workgroup(unsigned long long workgroups) {
    return workgroups <= kStripOneRoundWorkgroups ? kStripLateWorkgroup * kComputeUnits : 0u;
}

// Bit 2 of a chain's Params::reserved: the launch writes no more than kSmallOutputBytes (and has no segments that begin left of a row).
constexpr unsigned kSmallOutputBit = 4u;
// Whether a launch of the rows kernel takes the kernel for small outputs; run: elements a thread handles in a row (rows shorter than
// that, of which such a kernel knows nothing, are left to the other one), reserved: the parameter block's flags.
inline bool rows_small(unsigned w, unsigned run, unsigned reserved) { return (reserved & kSmallOutputBit) != 0u && w >= run; }

// Bit 3 of a chain's Params::reserved: the rows of every plane, read and written, follow each other without gaps, so the launch takes
// a plane as one row of w * h elements.
constexpr unsigned kFlatBit = 8u;
constexpr unsigned kFlatRun = 4;             // elements of a thread's run in such a launch
inline bool flat_fits(unsigned w, unsigned h) {
    const unsigned long long n = (unsigned long long)w * h;
    return n >= kFlatRun && n <= 0x7fff0000ull;
}
// The workgroups of a plane of such a launch; `rows`: segments of 64 runs per wave, of which a workgroup has four.
inline unsigned flat_blocks(unsigned w, unsigned h, unsigned reserved, unsigned rows) {
    const unsigned per_block = 64u * kFlatRun * 4u * rows;
    return unsigned(((unsigned long long)w * h + rows_phase_bound(reserved) + per_block - 1u) / per_block);
}

// Launches of the rows kernel with few workgroups (a single 1080p image is 1 080 of them at two rows per thread, about four per compute unit,
// so some units get five and some four) take half the rows, or segments, per thread: twice the workgroups spread evenly, which on such
// launches outweighs the shorter run of independent loads per thread.  The line, in workgroups (rows_few_blocks in the kernels' header): chains
// whose runs go through the LDS 2048, others 1024.  us with the line at 1024 / 2048: NV12 to float3 2000x1500 (1 504) 8.1 / 7.6, 2200x1200
// (1 350) 7.9 / 7.2, 1922x1082 (1 088) 6.7 / 6.4; RGB to NV12 1920x1080 (1 080) 3.4 / 3.6, 2560x1440 (1 800) 4.1 / 4.6; RGB to P010 1920x1080 4.6 / 4.9,
// 2000x1500 6.2 / 6.7.  Planes without gaps, with the line at 768 / 1024 / 2048: 4 uchar3 images of 1279x719 (1 800) 4.5 / 4.5 / 4.9, 4 of
// 849x880 (1 460; 4 launches) 16.2 / 16.2 / 17.9, 50 operations on 3840x2160 floats (2 025) 12.6 / 12.6 / 13.6; at 512: 4 of 1209x263 (624) 12.4 -> 13.05.
// Some chains below that line are faster with all their rows where those still make a round of two to four workgroups per compute unit (rows_keep_whole
// in the kernels' header): semi-planar video, and elements that go through the LDS at both ends.  us, all rows / half, 30 (20) buffers in turn: NV12 to
// float3 1280x720 (450) 3.44 / 3.45, 1280x960 (600) 3.94 / 4.00, 1536x1100 (828) 4.87 / 5.20, 1600x1000 (875) 5.06 / 5.15, 1792x1080 (945) 5.16 / 5.54, P010 to float3
// 5.43 / 5.88, 1922x1082 (1 088) 6.79 / 6.58; float3 squared, rows with gaps, 1024x600 (300) 3.81 / 3.67, 1280x960 6.55 / 6.91, 1600x800 (700) 6.59 / 7.58,
// 1792x1080 8.66 / 10.10, 2000x1300 (1 304) 14.2 / 13.0; without gaps 1280x960 6.55 / 6.71, 1792x1080 8.64 / 10.06.  Other chains are not:
// uchar3 to float3 1280x960 4.62 / 4.18, two fields of uchar3 to float3 1536x1100 6.01 / 5.38, float3 to uchar3 1536x1100 6.23 / 6.08.
constexpr unsigned kRowsFewBlocks = 1024, kRowsFewBlocksExchange = 2048, kRowsWholeFrom = 512, kRowsWholeTo = 1024;
// blocks: of a launch with all rows; few: rows_few_blocks of the chain.
inline constexpr bool rows_halved(unsigned long long blocks, unsigned few, bool keep_whole) {
    return blocks < few && !(keep_whole && blocks >= kRowsWholeFrom && blocks <= kRowsWholeTo);
}

// Which tiles a launch of the bilinear kernel's tile form takes: 128x8 pixels, or smaller ones where it would have few of those (per-wave
// latency, see the kernels' header).  us, tiles of 128x8 / 128x4 / 64x4 pixels (in brackets: how many of 128x8): NV12 to 148x85 (22)
// 3.23 / 2.41 / 2.09, to 320x180 (69) 2.58 / 2.05 / 1.94, to 400x300 (152) 3.23 / 2.61 / 2.69, to 1100x700 (792) 5.32 / 4.71 / 5.38, to 1333x800 (1100)
// 6.2 / 5.1 / 6.3, to 1600x900 (1469) 6.5 / 6.0 / 7.6, to 1920x1000 (1875) 7.6 / 6.7, to 2300x1300 (2934) 11.3 / 11.6; 5 thumbnails of 128x128 (80) 3.17 / 2.46 / 2.28, of 256x256 (320) 3.41 / 2.98 / 3.17; 8 crops
// to 64x64 (64) 2.96 / 2.38 / 2.16, to 224x64 (128) 3.09 / 2.42 / 2.63, to 224x224 (448) 3.73 / 3.46 / 3.99, to 300x200 (600) 4.07 / 3.89 / 4.34, to 384x300 (912)
// 4.60 / 4.42, to 320x320 (960) 4.56 / 4.77 / 5.59, 64 crops to 300x64 (1536) 5.9 / 6.3 / 8.0.  Reads with operations of their own under the resize cross later, cheap ones as well: uchar3 1920x1080
// with a cast fused, 128x8 / 128x4, to 1333x800 5.4 / 5.3, to 1400x900 (1243) 5.5 / 5.1, to 1600x900 5.4 / 5.4, to 1800x1000 (1875) 6.6 / 6.4, to 1920x1080 (2025) 6.1 /
// 5.7; cast, multiplication and addition 5.8 / 5.3, 6.0 / 5.5, 6.1 / 6.0, 7.4 / 7.0, 7.4 / 7.3.
constexpr unsigned kGatherFewTiles = 128, kGatherSomeTiles = 920, kGatherSomeTilesFused = 2560;
// A lane's pixels along x and a wave's rows: form 0 has the kernels' own (FKD_GATHER_XI, FKD_GATHER_YI), 1 and 2 are named by theirs.
inline constexpr unsigned gather_form_xi(unsigned form, unsigned own) { return form != 0u ? form : own; }
inline constexpr unsigned gather_form_yi(unsigned form, unsigned own) { return form != 0u ? 1u : own; }
inline unsigned gather_form(unsigned w, unsigned h, unsigned planes, unsigned some_tiles) {
    const unsigned long long tiles = (unsigned long long)((w + 127u) / 128u) * ((h + 7u) / 8u) * planes;
    return tiles < kGatherFewTiles ? 1u : tiles < some_tiles ? 2u : 0u;
}

// Bit 4 of a chain's Params::reserved: a launch of the bilinear kernel whose stores are moved on to line boundaries (lines_pay, LineStores in
// the kernels' header): workgroups of eight rows of 32 lanes or of four rows of 64.  Wide rows have 64; narrow ones too where the launch would
// have few workgroups (8 crops to 250x250, 256 of them: 4.5 us with 32 lanes, 3.7 with 64; 64 crops to 193x105, 896: 6.2 / 6.7).
constexpr unsigned kLinesBit = 16u, kLinesWidth = 640;
inline constexpr unsigned lines_lanes(unsigned w, unsigned h, unsigned planes) {
    return w > 256u || (unsigned long long)((h + 7u) / 8u) * planes < 540u ? 64u : 32u;
}

// Rows of a workgroup of the bilinear kernel's strip form: half a wave each.
constexpr unsigned kStripFormRows = 8;

// Workgroup x of the gx of plane z, one row of workgroups per plane, as the number of its part of the plane: the hardware deals workgroups round-robin
// to the 8 XCDs, so x is on XCD (z * gx + x) % 8, and XCD k takes the k-th run of parts, which share source lines, in every plane.
inline constexpr unsigned plane_band(unsigned x, unsigned gx, unsigned z) {
    const unsigned first = z * gx % 8u, k = (first + x) % 8u;
    const unsigned longer = ((1u << gx % 8u) - 1u) << first;           // the XCDs with one workgroup more, round the end
    return k * (gx / 8u) + unsigned(__builtin_popcount((longer | longer >> 8) & ((1u << k) - 1u))) + x / 8u;
}

// What the launcher of a run-time compiled kernel needs to know about it; the kernel's module publishes one.
struct JitMeta {
    unsigned gather;          // 1: gather kernel geometry, 0: rows kernel geometry
    unsigned params_bytes;    // sizeof(Chain::Params)
    unsigned v, rows;         // rows kernel: elements per thread along x, rows per thread
    unsigned xi, yi, by;      // gather kernel: pixels per lane along x, rows per wave, waves per workgroup
    unsigned max_planes;      // most planes (grid z) a launch may have, 0: no limit of the kernel's own
    unsigned strip_width;     // gather kernel: outputs up to this width are launched in strip form (TileGeom::tiles_x == 0), 0: never
    unsigned bands;           // rows kernel: 1 when launches of kRowsBandBlocks blocks per plane or more take the bands form of grid, 2 when smaller ones may as well (rows_bands_2d)
    unsigned has_small;       // rows kernel: 1 when the module has a kernel for small outputs (see rows_small)
    unsigned has_flat;        // rows kernel: 1 when the module has kernels for planes taken as one row (kFlatBit)
    unsigned stream_bytes;    // gather kernel with a planar writer: bytes stored per output element (see kStreamOutputBytes), else 0
    unsigned some_tiles;      // gather kernel: the last argument of gather_form
    unsigned few_blocks;      // rows kernel: rows_few_blocks
    unsigned keep_whole;      // rows kernel: rows_keep_whole
};

// Which of a run-time compiled module's kernels a launch takes, and its grid of workgroups of 64 lanes by block_y waves.  active: the extents and
// flags the parameter block begins with; strip: whether the strip form may be taken.  (The constants a module was compiled with are the
// module's own: everything here comes from its JitMeta.)
struct JitGeometry {
    const char *kernel, *form;            // see LaunchInfo
    unsigned which;                       // 0 the chain's own kernel, 1 to 6 those of jit_other_body
    unsigned long long grid_x;
    unsigned grid_y, block_y;
    TileGeom g;
};
inline JitGeometry jit_geometry(const JitMeta& m, const unsigned (&active)[4], bool strip) {
    JitGeometry l{m.gather ? "gather_jit" : "rows_jit", m.gather ? "tiles" : (m.max_planes != 0u ? "divergent" : "rows"), 0u, 0u, 1u, m.gather ? m.by : 4u, TileGeom{0, 0, 0, 0}};
    const unsigned w = active[0], h = active[1], planes = active[2], flags = active[3];
    const bool streamed = m.gather && (unsigned long long)w * h * planes * m.stream_bytes > kStreamOutputBytes;
    strip = strip && m.gather && m.strip_width != 0u && w != 0u;
    if (strip && (flags & kLinesBit) != 0u) {
        // (rows of 64 lanes only)
        l.kernel = (flags & 1u) != 0u ? "strip_jit" : "gather_jit";
        l.form = "strip_lines";
        l.which = 3u;
        l.grid_x = (h + 3u) / 4u;
        l.g.n_tiles = streamed ? kStreamFlag : 0u;
    } else if (strip && w <= m.strip_width && (flags & 1u) != 0u) {
        // strip form: tiles_x == 0 tells the kernel, and n_tiles carries the launch's priority schedule
        l.kernel = "strip_jit";
        l.form = "strip";
        l.grid_x = (h + kStripFormRows - 1u) / kStripFormRows;
        l.g.n_tiles = strip_first_late_workgroup(l.grid_x * planes) | (streamed ? kStreamFlag : 0u) | ((flags & 2u) != 0u ? kAnyPitchFlag : 0u);
    } else if (m.gather) {
        l.which = gather_form(w, h, planes, m.some_tiles);
        const unsigned tw = 64u * gather_form_xi(l.which, m.xi), th = m.by * gather_form_yi(l.which, m.yi);
        l.g.tiles_x = (w + tw - 1u) / tw;
        l.g.tiles_y = (h + th - 1u) / th;
        l.g.n_tiles = streamed ? kStreamFlag : 0u;       // (the kernel counts its tiles itself)
        l.g.tiles_x_magic = division_magic(l.g.tiles_x, l.g.tiles_x * l.g.tiles_y);
        l.grid_x = (l.g.tiles_x * l.g.tiles_y + 7u) / 8u * 8u;
    } else if (m.has_flat != 0u && (flags & kFlatBit) != 0u) {
        l.form = "flat";
        l.which = 2u;
        l.grid_x = flat_blocks(w, h, flags, m.rows);
        const bool few = m.rows > 1u && rows_halved(l.grid_x * planes, m.few_blocks, m.keep_whole != 0u);
        if ((flags & kSmallOutputBit) != 0u || few) {
            l.which = (flags & kSmallOutputBit) != 0u ? 3u : 5u;
            if (m.rows > 1u) l.grid_x = flat_blocks(w, h, flags, m.rows / 2u);
        }
    } else {
        if (m.has_small != 0u && rows_small(w, m.v, flags)) l.which = 1u;
        unsigned rows = m.rows;
        if (m.max_planes == 0u && m.rows > 1u) {
            const bool few = rows_halved((unsigned long long)((w + 64u * m.v - 1u) / (64u * m.v)) * ((h + 4u * rows - 1u) / (4u * rows)) * planes, m.few_blocks, m.keep_whole != 0u);
            if (l.which == 0u && few) l.which = 4u;
            if (l.which == 1u && !few) l.which = 6u;
            if (few) rows /= 2u;
        }
        const unsigned gx = (w + (m.max_planes != 0u ? 0u : rows_phase_bound(flags)) + 64u * m.v - 1u) / (64u * m.v), gy = (h + 4u * rows - 1u) / (4u * rows);
        l.grid_x = gx;
        l.grid_y = gy;
        const bool bands = m.bands && (unsigned long long)gx * gy >= kRowsBandBlocks;
        if (bands || (m.bands > 1u && rows_bands_2d(gx, gy))) {
            l.g.tiles_x = gx;
            l.g.tiles_y = gy;
            l.g.tiles_x_magic = division_magic(gx, gx * gy);
        }
        if (bands) {
            // as launch_rows_with: one-dimensional, eight equal runs of the plane's blocks
            l.g.n_tiles = gx * gy * planes;
            l.grid_x = ((unsigned long long)gx * gy + 7u) / 8u * 8u;
            l.grid_y = 1u;
        }
    }
    return l;
}

} // namespace fkd
