// fkd_launch.hpp -- host-side launchers of the ahead-of-time compiled kernels (grid geometry, host-side alignment
// check, hipLaunchKernel).  Launch geometry being replaced: FK/core/execution_model/executors.h:242-351.
#pragma once

#include "fkd_kernels.hpp"
#include "registry.hpp"

namespace fkd {

// ---- host-side launchers -------------------------------------------------------------------------------

// Launch with pointers to the arguments: the runtime then makes the only copy of the (up to 8 KB) parameter block,
// straight into its kernel-argument buffer; the <<< >>> form would first copy it by value onto this thread's stack.
template <class Kernel, class... Args>
inline hipError_t launch_by_pointer(Kernel kernel, dim3 grid, dim3 block, hipStream_t stream, const Args&... args) {
    void* ptrs[] = {const_cast<void*>(static_cast<const void*>(&args))...};
    return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, ptrs, 0, stream);
}

inline const char* aligned_name(bool aligned) { return aligned ? "rows" : "rows_unaligned"; }

template <class Chain, int V, int ROWS>
hipError_t launch_rows_with(const typename Chain::Params& p, hipStream_t stream, LaunchInfo* info, bool aligned) {
    const unsigned gx = (p.active_w + rows_phase_bound(p.reserved) + kRowsBX * V - 1) / (kRowsBX * V);
    const unsigned gy = (p.active_h + kRowsBY * ROWS - 1) / (kRowsBY * ROWS);
    dim3 grid(gx, gy, p.active_z);
    const dim3 block(kRowsBX, kRowsBY, 1);
    TileGeom g{};
    if constexpr (rows_in_bands<Chain>()) {
        // gathering reads, larger launches: a one-dimensional grid whose workgroups the kernel renumbers into one band per XCD
        if ((unsigned long long)gx * gy > 0x7fffff00ull) return hipErrorInvalidConfiguration;
        if (gx * gy >= kRowsBandBlocks) {
            grid = dim3(rows_band_chunk(gx * gy) * 8u, 1, p.active_z);
            g = TileGeom{gx, gy, gx * gy * p.active_z, division_magic(gx, gx * gy)};
        } else if (rows_by_points<Chain, V, ROWS>() && rows_bands_2d(gx, gy)) {
            g = TileGeom{gx, gy, 0u, division_magic(gx, gx * gy)};
        }
    }
    if (info) *info = LaunchInfo{aligned_name(aligned), {grid.x, grid.y, grid.z}, {block.x, block.y, 1}, 0, "rows"};
    if (grid.x == 0 || grid.y == 0 || grid.z == 0) return hipSuccess;
    if (grid.y > 65535u || grid.z > 65535u) return hipErrorInvalidConfiguration;
    const bool small = rows_small(p.active_w, V, p.reserved);
    if constexpr (!rows_any_x<Chain>(V)) {
        if (aligned) {
            if (small) return launch_by_pointer(&k_rows<Chain, V, ROWS, true, kRowsSmall>, grid, block, stream, p, g);
            return launch_by_pointer(&k_rows<Chain, V, ROWS, true, kRowsLines>, grid, block, stream, p, g);
        }
    }
    if (small) return launch_by_pointer(&k_rows<Chain, V, ROWS, false, kRowsSmall>, grid, block, stream, p, g);
    return launch_by_pointer(&k_rows<Chain, V, ROWS, false, kRowsLines>, grid, block, stream, p, g);
}

template <class Chain, int V, int ROWS>
hipError_t launch_flat(const typename Chain::Params& p, hipStream_t stream, LaunchInfo* info) {
    const unsigned blocks = flat_blocks(p.active_w, p.active_h, p.reserved, ROWS);
    if constexpr (ROWS > 1) {
        if (rows_halved((unsigned long long)blocks * p.active_z, rows_few_blocks<Chain>(), rows_keep_whole<Chain>())) return launch_flat<Chain, V, ROWS / 2>(p, stream, info);
    }
    const dim3 grid(blocks, 1, p.active_z), block(kRowsBX, kRowsBY, 1);
    if (info) *info = LaunchInfo{"rows", {grid.x, 1, grid.z}, {block.x, block.y, 1}, 0, "flat"};
    if (grid.z == 0) return hipSuccess;
    if (grid.z > 65535u) return hipErrorInvalidConfiguration;
    if ((p.reserved & kSmallOutputBit) != 0u) return launch_by_pointer(&k_flat<Chain, V, ROWS, true>, grid, block, stream, p);
    return launch_by_pointer(&k_flat<Chain, V, ROWS, false>, grid, block, stream, p);
}

template <class Chain>
hipError_t launch_rows(const typename Chain::Params& p, hipStream_t stream, LaunchInfo* info) {
    constexpr int V = RowsConfig<Chain>::V, ROWS = RowsConfig<Chain>::ROWS;
    if constexpr (rows_flat<Chain>()) {
        if ((p.reserved & kFlatBit) != 0u) return launch_flat<Chain, V, ROWS>(p, stream, info);
    }
    // Chains whose reads may start anywhere in a row have one kernel for rows at every alignment.  The others have one for rows
    // that all start on dword boundaries (checked here, once per launch, on the host) and one for the rest.
    bool aligned = true;
    if constexpr (!rows_any_x<Chain>(V)) aligned = Chain::Read::rows_aligned(p.read, 0) && Chain::Write::rows_aligned(p.write);
    if constexpr (ROWS > 1) {
        const unsigned long long gx = (p.active_w + kRowsBX * V - 1) / (kRowsBX * V);
        const unsigned long long gy = (p.active_h + kRowsBY * ROWS - 1) / (kRowsBY * ROWS);
        if (rows_halved(gx * gy * p.active_z, rows_few_blocks<Chain>(), rows_keep_whole<Chain>())) return launch_rows_with<Chain, V, ROWS / 2>(p, stream, info, aligned);
    }
    return launch_rows_with<Chain, V, ROWS>(p, stream, info, aligned);
}

template <class Chain>
hipError_t launch_gather(const typename Chain::Params& p, hipStream_t stream, LaunchInfo* info) {
    constexpr int XI = FKD_GATHER_XI, YI = FKD_GATHER_YI;
    constexpr bool kStreams = writer_streams<Chain>();
    const bool streamed = kStreams && (unsigned long long)p.active_w * p.active_h * p.active_z * sizeof(typename Chain::Value) > kStreamOutputBytes;
    if constexpr (strip_capable<Chain>()) {
        if (p.active_w != 0 && (p.reserved & kLinesBit) != 0u && fklhip::strip_enabled()) {
            const unsigned lanes = lines_lanes(p.active_w, p.active_h, p.active_z), rows = kStripThreads / lanes;
            const dim3 grid((p.active_h + rows - 1) / rows, 1, p.active_z), block(kGatherBX, kStripThreads / kGatherBX, 1);
            if (info) *info = LaunchInfo{(p.reserved & 1u) != 0u ? "strip" : "gather", {grid.x, 1, grid.z}, {block.x, block.y, 1}, unsigned((lanes == 32u ? 9 * 32 : 11 * 64) * 16 + (kStripThreads / 64) * 4), "strip_lines"};
            if (grid.x == 0 || grid.z == 0) return hipSuccess;
            if (grid.z > 65535u) return hipErrorInvalidConfiguration;
            if (lanes == 32u) {
                if (streamed) return launch_by_pointer(&k_strip_lines<Chain, kStreams, 32>, grid, block, stream, p);
                return launch_by_pointer(&k_strip_lines<Chain, false, 32>, grid, block, stream, p);
            }
            if (streamed) return launch_by_pointer(&k_strip_lines<Chain, kStreams, 64>, grid, block, stream, p);
            return launch_by_pointer(&k_strip_lines<Chain, false, 64>, grid, block, stream, p);
        }
        // Narrow outputs (batches of small planes): the strip form, whose workgroups own 8 whole rows of a plane.
        // (an output without columns has no workgroup in the tile form's grid: it falls through and launches nothing)
        if (p.active_w != 0 && p.active_w <= unsigned(kStripMaxWidth) && (p.reserved & 1u) != 0 && fklhip::strip_enabled()) {
            const dim3 grid((p.active_h + kStripRows - 1) / kStripRows, 1, p.active_z), block(kGatherBX, kStripThreads / kGatherBX, 1);
            if (info) *info = LaunchInfo{"strip", {grid.x, 1, grid.z}, {block.x, block.y, 1}, unsigned(kStripMaxWidth * 16 + (kStripThreads / 64) * 4), "strip"};
            if (grid.x == 0 || grid.z == 0) return hipSuccess;
            if (grid.z > 65535u) return hipErrorInvalidConfiguration;
            const unsigned first_late = strip_first_late_workgroup((unsigned long long)grid.x * grid.z);
            if ((p.reserved & Chain::kStripAnyPitch) != 0u) {
                if (streamed) return launch_by_pointer(&k_strip<Chain, kStreams, true>, grid, block, stream, p, first_late);
                return launch_by_pointer(&k_strip<Chain, false, true>, grid, block, stream, p, first_late);
            }
            if (streamed) return launch_by_pointer(&k_strip<Chain, kStreams, false>, grid, block, stream, p, first_late);
            return launch_by_pointer(&k_strip<Chain, false, false>, grid, block, stream, p, first_late);
        }
    }
    const unsigned form = gather_form(p.active_w, p.active_h, p.active_z, gather_some_tiles<Chain>());
    const unsigned TW = kGatherBX * gather_form_xi(form, XI), TH = kGatherBY * gather_form_yi(form, YI);
    TileGeom g;
    g.tiles_x = (p.active_w + TW - 1) / TW;
    g.tiles_y = (p.active_h + TH - 1) / TH;
    g.n_tiles = g.tiles_x * g.tiles_y * p.active_z;
    g.tiles_x_magic = division_magic(g.tiles_x, g.tiles_x * g.tiles_y);
    const unsigned chunk = (g.tiles_x * g.tiles_y + 7u) / 8u;
    const dim3 grid(chunk * 8u, 1, p.active_z), block(kGatherBX, kGatherBY, 1);
    if (info) *info = LaunchInfo{"gather", {grid.x, 1, grid.z}, {block.x, block.y, 1}, 0, "tiles"};
    if (g.n_tiles == 0) return hipSuccess;
    if (grid.z > 65535u) return hipErrorInvalidConfiguration;
    if (form == 1u) return launch_by_pointer(&k_gather<Chain, 1, 1, false>, grid, block, stream, p, g);
    if (form == 2u) return launch_by_pointer(&k_gather<Chain, 2, 1, false>, grid, block, stream, p, g);
    if (streamed) return launch_by_pointer(&k_gather<Chain, XI, YI, kStreams>, grid, block, stream, p, g);
    return launch_by_pointer(&k_gather<Chain, XI, YI, false>, grid, block, stream, p, g);
}

// Several chains in one launch: the grid of the rows kernel over the largest extent, alignment decided per plane on
// the device.
template <class D>
hipError_t launch_divergent(const typename D::Params& p, hipStream_t stream, LaunchInfo* info) {
    constexpr int V = RowsConfig<D>::V, ROWS = RowsConfig<D>::ROWS;
    const unsigned gx = (p.active_w + kRowsBX * V - 1) / (kRowsBX * V);
    const unsigned gy = (p.active_h + kRowsBY * ROWS - 1) / (kRowsBY * ROWS);
    const dim3 grid(gx, gy, p.active_z), block(kRowsBX, kRowsBY, 1);
    if (info) *info = LaunchInfo{"divergent", {grid.x, grid.y, grid.z}, {block.x, block.y, 1}, 0, "divergent"};
    if (grid.x == 0 || grid.y == 0 || grid.z == 0) return hipSuccess;
    if (grid.y > 65535u || grid.z > unsigned(D::kMaxPlanes)) return hipErrorInvalidConfiguration;
    return launch_by_pointer(&k_divergent<D>, grid, block, stream, p);
}

template <class Chain>
hipError_t launch_chain(const typename Chain::Params& p, hipStream_t stream, LaunchInfo* info) {
    if constexpr (IsDivergent<Chain>::value) return launch_divergent<Chain>(p, stream, info);
    else if constexpr (is_gather_chain<Chain>()) return launch_gather<Chain>(p, stream, info);
    else return launch_rows<Chain>(p, stream, info);
}

} // namespace fkd
