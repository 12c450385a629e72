// fkd/launch_info.hpp -- what a launcher reports about the launch it made, and the geometry it hands to the kernels:
// shared by the launchers of the ahead-of-time kernels, the launcher of the run-time compiled ones and the kernels
// themselves (plain C++, no HIP).
#pragma once

namespace fkd {

struct LaunchInfo {
    const char* kernel;   // "rows", "rows_unaligned" (chains with a kernel of its own for such rows), "gather" or "strip"
    unsigned grid[3], block[3];
    unsigned lds_bytes;
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
// the stores alone take 55 us either way.  The line lies where the two cross (64 crops of a 1920x1080 image; written through /
// non-temporal): 224x224, 38 MB 9.8 / 10.2 us; 288x288, 64 MB 14.4 / 14.6; 320x320, 79 MB 17.2 / 16.4; 384x384, 113 MB 26.9 /
// 21.6; 512x512, 201 MB 48.8 / 35.1.
constexpr unsigned long long kStreamOutputBytes = 64ull << 20;
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

// What the launcher of a run-time compiled kernel needs to know about it; the kernel's module publishes one.
struct JitMeta {
    unsigned gather;          // 1: gather kernel geometry, 0: rows kernel geometry
    unsigned params_bytes;    // sizeof(Chain::Params)
    unsigned v, rows;         // rows kernel: elements per thread along x, rows per thread
    unsigned xi, yi, by;      // gather kernel: pixels per lane along x, rows per wave, waves per workgroup
    unsigned max_planes;      // most planes (grid z) a launch may have, 0: no limit of the kernel's own
    unsigned strip_width;     // gather kernel: outputs up to this width are launched in strip form (TileGeom::tiles_x == 0), 0: never
    unsigned bands;           // rows kernel: 1 when launches of kRowsBandBlocks blocks per plane or more take the bands form of grid
    unsigned stream_bytes;    // gather kernel with a planar writer: bytes stored per output element (see kStreamOutputBytes), else 0
};

} // namespace fkd
