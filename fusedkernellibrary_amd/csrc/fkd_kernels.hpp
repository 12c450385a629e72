// fkd_kernels.hpp -- the gfx950 kernel skeletons of the fused data-parallel path and their launchers.
//
// Two skeletons cover every chain; which one a chain gets is decided from its read operation at compile time.
//
//  rows kernel    one thread produces V = 4 horizontally adjacent outputs of one row of plane z.  Reads and
//                 writes of 4 elements move as dwordx3 / dwordx4 accesses (12 bytes for uchar3, 16 for float,
//                 48 for float3) that consecutive lanes make contiguous, so a wave64 touches whole cache lines;
//                 rows may start at any byte and have any width.
//                 Each thread handles ROWS rows so several independent loads are in flight per lane.
//                 Plane z = workgroup index in z: horizontal (batch) fusion, per-plane parameters are wave
//                 uniform and come out of the kernel-argument segment through scalar loads.
//
//  gather kernel  for chains whose read is a bilinear resize: a workgroup owns a tile of the output of one plane,
//                 a wave owns whole output rows of it, so source rows, vertical weights and all row addresses are
//                 wave uniform (scalar registers); a lane reads the four taps of each of its pixels straight from
//                 global memory as whole elements at byte granularity.  Whatever was fused into the read (colour
//                 conversion, per-plane arithmetic) is applied per tap, in the reference's order.  Workgroups are
//                 renumbered so each XCD works on a contiguous run of a plane's tiles and its L2 sees the source
//                 rows those tiles share.
//
// Reference being replaced: TransformDPP<GPU_NVIDIA>::exec and launchTransformDPP_Kernel,
// FK/core/execution_model/data_parallel_patterns.h:223-242 and executor_details/executor_kernels.h:26-30;
// launch geometry FK/core/execution_model/executors.h:242-351.
#pragma once

#if !defined(__HIPCC_RTC__)
#include <hip/hip_runtime.h>   // the run-time compiler provides the HIP device API without any header
#endif

#include <fkd/launch_info.hpp>
#include <fkd/ops.hpp>

namespace fkd {

template <int I> struct IntTag { static constexpr int value = I; };

// ---- chain classification ---------------------------------------------------------------------------

template <class R> struct ResizeRoot { static constexpr bool value = false; };
template <int AR, class Back> struct ResizeRoot<ResizeLinear<AR, Back>> {
    static constexpr bool value = true;
    static constexpr bool batched = false;
    using Resize = ResizeLinear<AR, Back>;
};
template <int N, int AR, class Back> struct ResizeRoot<BatchRead<N, ResizeLinear<AR, Back>>> {
    static constexpr bool value = true;
    static constexpr bool batched = true;
    using Resize = ResizeLinear<AR, Back>;
};

template <int N, int AR, class Back> struct ResizeRoot<BatchReadDefault<N, ResizeLinear<AR, Back>>> {
    static constexpr bool value = true;
    static constexpr bool batched = true;
    using Resize = ResizeLinear<AR, Back>;
};
template <class R> struct HasDefaultPlanes { static constexpr bool value = false; };
template <int N, class PlaneOp> struct HasDefaultPlanes<BatchReadDefault<N, PlaneOp>> { static constexpr bool value = true; };

// Reads whose taps are scattered gathers (warps).
template <class R> constexpr bool is_scattered_read() {
    if constexpr (requires { R::kGatherRead; }) return R::kGatherRead;
    else if constexpr (requires { typename R::Plane; }) return is_scattered_read<typename R::Plane>();
    else return false;
}

template <class Chain> constexpr bool is_gather_chain() {
    if constexpr (ResizeRoot<typename Chain::Read>::value)
        return ResizeRoot<typename Chain::Read>::Resize::BackOp::kTapCursor;
    else
        return false;
}

// Stores of a lane-masking writer (kLaneMasked); other writers never reach these calls, the indirection only keeps their
// instantiations from looking the members up.
template <class WP, class Plane> __device__ __forceinline__ u32 masked_row_offset(int y, const Plane& plane) {
    if constexpr (requires { WP::kLaneMasked; }) return WP::row_offset(y, plane); else return 0u;
}
template <class WP, bool STREAM, class Plane, class V> __device__ __forceinline__ void masked_put(const Plane& plane, u32 row_off, u32 lane_off, const V& v) {
    if constexpr (requires { WP::kLaneMasked; }) WP::template put_masked<STREAM>(plane, row_off, lane_off, v);
}
// Whether the chain's writer has a streaming form (see kStreamOutputBytes) for the bilinear kernel to choose.
template <class Chain> constexpr bool writer_streams() {
    if constexpr (requires { Chain::Write::Plane::kLaneMasked; }) return Chain::Write::Plane::kLaneMasked; else return false;
}

// (The geometry a launcher hands to kernels that renumber their workgroups -- TileGeom, division_magic, the limits that
// choose a form of grid -- is in fkd/launch_info.hpp, which the launchers of run-time compiled kernels share.)

// ---- rows kernel ---------------------------------------------------------------------------------------

constexpr int kRowsBX = 64;   // lanes along x: one wave per row segment
constexpr int kRowsBY = 4;    // waves per workgroup
constexpr unsigned long long kStreamElements = 1ull << 26;   // launches over more elements stream their input

// For the test of what run-time compilation does with a chain whose per-thread array cannot stay in registers: with
// FKD_TEST_UNRESOLVED_INDEX defined, the rows kernel indexes its values with an offset that is zero when the kernel runs
// but unknown when it is compiled (an index the optimiser cannot resolve keeps the array in memory).  Zero otherwise.
#ifdef FKD_TEST_UNRESOLVED_INDEX
#define FKD_TEST_INDEX_OFFSET int(p.reserved >> 31)
#else
#define FKD_TEST_INDEX_OFFSET 0
#endif

// One wave's part of the rows kernel: V elements of each of ROWS rows per lane, row r from element x[r] on.  MODE as in
// detail::load_run for the loads; PLAIN: stores without the non-temporal hint.
// EDGE: the wave's segment of 64 * V elements, which begins at seg[r], reaches past the end of the row
// (kRowEnd: lanes that have no element inside are not here) or past either end (kRowEnds: all lanes of the wave are here).  A
// lane that has fewer than V of its elements inside, or none, then works on the first or last V elements of the row, and only
// the elements of the segment are stored; what a lane reads beside its own is not used or its neighbour's in the same wave,
// so a chain that works in place is none the wiser.
// kEvenWidth beside them, for reads whose runs are at their best from even elements: the row's width is even, so the last V elements
// begin at an even one too and no lane has to be asked (asked row by row, a thread's second row was fetched behind its first:
// P010 to RGB at 244x262 2.41 instead of 2.15 us, at 1036x744 4.34 instead of 3.97).
constexpr int kRowEnd = 1, kRowEnds = 2, kEvenWidth = 4;
template <class Chain, int V, int ROWS, int MODE, bool PLAIN, int EDGE_BITS = 0>
__device__ __forceinline__ void rows_full(const typename Chain::Params& p, u32 kernarg_offset, const int (&seg)[ROWS], const int (&x)[ROWS],
                                          int ybase, int z, int aw, int ah) {
    using R = typename Chain::Read;
    using W = typename Chain::Write;

    // All loads first, unconditionally (rows past the end re-read the last row, which is in bounds), so every
    // lane has ROWS independent wide loads in flight before the first use; only the stores are predicated.
    constexpr int EDGE = EDGE_BITS & 3;
    constexpr bool EVEN = (EDGE_BITS & kEvenWidth) != 0;
    Slot<typename R::Out> in[ROWS * V];
    int x0[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const int y = ybase + r < ah ? ybase + r : ah - 1;
        x0[r] = x[r];
        if constexpr (EDGE == kRowEnd) x0[r] = x[r] < aw - V ? x[r] : aw - V;
        if constexpr (EDGE == kRowEnds) x0[r] = x[r] < 0 ? 0 : (x[r] < aw - V ? x[r] : aw - V);
        if constexpr (EVEN) x0[r] &= ~1;                                  // (even already: said to the compiler)
        Slot<typename R::Out> row[V];
        R::template exec_row<V, MODE>(x0[r], y, z, p.read, row);
#pragma unroll
        for (int i = 0; i < V; ++i) in[r * V + i].v = row[i].v;
    }
    // all ROWS*V elements go through the chain together, operation by operation
    Slot<typename Chain::Value> out[ROWS * V];
    if constexpr (Chain::kLongChain) Chain::template compute_run_kernarg<ROWS * V>(in, out, (const FKD_CONSTANT char*)__builtin_amdgcn_kernarg_segment_ptr() + kernarg_offset);
    else Chain::template compute_run<ROWS * V>(in, out, p.ops);
    constexpr int STORE = MODE | (PLAIN ? detail::kPlainStores : 0);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const int y = ybase + r;
        Slot<typename Chain::Value> row[V];
#pragma unroll
        for (int i = 0; i < V; ++i) row[i].v = out[r * V + i + FKD_TEST_INDEX_OFFSET].v;
        if (y >= ah) continue;
        if constexpr (EDGE == kRowEnds && has_edge_store<W, V>()) {
            W::template exec_edge<V>(seg[r], x0[r], aw, y, z, row, p.write);
        } else if constexpr (EDGE != 0) {
            if (x0[r] == x[r]) {
                W::template exec_row<V, STORE>(x0[r], y, z, row, p.write);
            } else if (EDGE == kRowEnd || (x[r] > -V && x[r] < aw)) {
#pragma unroll
                for (int i = 0; i < V; ++i) {
                    if (EDGE == kRowEnd && i == 0) continue;              // (the first of the row's last V is never the lane's)
                    if (x0[r] + i >= x[r] && (EDGE == kRowEnd || x0[r] + i < x[r] + V)) W::exec(x0[r] + i, y, z, row[i].v, p.write);
                }
            }
        } else {
            W::template exec_row<V, STORE>(x0[r], y, z, row, p.write);
        }
    }
}

// Whether waves may take runs that start anywhere in a row.
template <class Chain> constexpr bool rows_any_x(int v) { return v > 1 && any_x<typename Chain::Read>(); }

// Chains whose read gathers its taps from wherever the coordinates fall (warps, bilinear reads without a tap cursor): their
// larger launches number the workgroups of a plane so that each XCD works on a contiguous band of the output.
template <class Chain> constexpr bool rows_in_bands() {
    return ResizeRoot<typename Chain::Read>::value || is_scattered_read<typename Chain::Read>();
}
// The workgroups of a plane, bands form: the grid is one-dimensional, 8 * ceil(blocks / 8) workgroups per plane.  The
// hardware deals consecutive workgroup numbers round-robin to the 8 XCDs; XCD k takes the k-th contiguous eighth of the
// plane's blocks (row-major), so that neighbouring blocks, whose taps share source lines, share an L2.  With the
// workgroups in plain row-major order a warp fetched its source 2.5 to 3.2 times, once into nearly every L2; in bands it
// is fetched once (rocprofv3 FETCH_SIZE), and a 3840 x 2160 warp takes 25.1 instead of 30.8 us.  Launches of fewer than
// kRowsBandBlocks blocks per plane keep the two-dimensional grid; those of warps by columns are renumbered into bands inside it
// (rows_bands_2d).  (rows_band_chunk and kRowsBandBlocks: fkd/launch_info.hpp.)

// `kernarg_offset`: where p sits inside the kernel-argument segment (0 when the chain's parameter block is the
// kernel's first argument); long chains fetch their operations' parameters from there.  BANDS: the launch has the bands
// form of grid (see rows_band_chunk).
// FORM: kRowsOpen serves every launch; kRowsLines as well, one whose grid has room for segments that begin left of a row
// (Chain::row_phase_bound); kRowsSmall those of rows_small.  The latter is a kernel of its own, a third to a fifth as long: besides the
// stores' hint (see kSmallOutputBytes) small launches lost 2 to 5 % to the length of the other one (30 operations on 1544x90 floats
// 2.31 us instead of 2.20).  Larger launches gain nothing from shorter kernels of their own (50 operations at 3840x2160 12.1 -> 12.3 us, RGB
// to NV12 6.9 -> 7.0).
constexpr int kRowsOpen = 0, kRowsLines = 1, kRowsSmall = 2;
template <class Chain, int V, int ROWS, bool ALIGNED, bool BANDS = false, int FORM = kRowsOpen>
__device__ __forceinline__ void rows_body(const typename Chain::Params& p, u32 kernarg_offset = 0, const TileGeom* bands = nullptr) {
    using R = typename Chain::Read;
    using W = typename Chain::Write;
    const int z = blockIdx.z;
    const int aw = int(p.active_w), ah = int(p.active_h);
    u32 block_x = blockIdx.x, block_y = blockIdx.y;
    if constexpr (BANDS) {
        // (blocks per row and per column, and the multiplier that divides by the former, come from the launcher, which
        // leaves them zero for a two-dimensional grid; wave uniform)
        const u32 gx = bands->tiles_x, blocks = gx * bands->tiles_y;
        if (blocks != 0u) {
            const u32 tin = (blockIdx.x % 8u) * rows_band_chunk(blocks) + blockIdx.x / 8u;
            if (tin >= blocks) return;
            block_y = bands->tiles_x_magic ? u32(((unsigned long long)tin * bands->tiles_x_magic) >> 32) : tin / gx;
            block_x = tin - block_y * gx;
        }
    }
    // Wave-cooperative accesses (mode 2 of load_run / store_run) need every lane of the wave on a full run.
    constexpr bool kExchange = (detail::wave_exchange_ok<typename R::Out>(V) || detail::wave_exchange_ok<typename W::In>(V));
    // A launch over more elements than the last-level cache could hold between two launches reads them with the
    // non-temporal hint (100 images of 1920x1080 uchar3: 225 -> 209 us); smaller inputs are left to the caches, where a
    // pipeline's previous stage may have put them (the hint costs 15 % on a 33 MB image that is still cached).
    constexpr bool kSmall = FORM == kRowsSmall;
    constexpr bool kMayStream = !kSmall && !Chain::kLongChain && !kExchange;
    const bool stream = kMayStream && (unsigned long long)(u32(aw)) * u32(ah) * gridDim.z > kStreamElements;
    if constexpr (rows_any_x<Chain>(V)) {
        // A wave owns a segment of 64 * V elements of a row.  Segments are counted from the row's start or, in launches with
        // room for it (row_phase_bound), from the last line boundary before it, so that every wave but the two at a row's ends
        // stores whole lines: a line shared by two waves leaves the chip as two partial writes.
        if (kSmall || aw >= V) {
            const int yw = (block_y * kRowsBY + __builtin_amdgcn_readfirstlane(int(threadIdx.y))) * ROWS;
            if (yw >= ah) return;
            constexpr int kWhole = kExchange ? 2 | detail::kAnyAlign : 0;
            int seg[ROWS], x[ROWS];
            bool whole = true;
            auto go = [&](auto edge_tag) {
                constexpr int EDGE = decltype(edge_tag)::value;
                if constexpr (kMayStream) {
                    if (stream) { rows_full<Chain, V, ROWS, (EDGE ? 0 : kWhole) | 4, false, EDGE>(p, kernarg_offset, seg, x, yw, z, aw, ah); return; }
                }
                if constexpr (EDGE != 0 && x_group<R>() == 2 && V % 2 == 0) {
                    if ((aw & 1) == 0) { rows_full<Chain, V, ROWS, 0, kSmall, EDGE | kEvenWidth>(p, kernarg_offset, seg, x, yw, z, aw, ah); return; }
                }
                rows_full<Chain, V, ROWS, EDGE ? 0 : kWhole, kSmall, EDGE>(p, kernarg_offset, seg, x, yw, z, aw, ah);
            };
            if constexpr (FORM == kRowsLines && has_row_phase<W>()) {
                const u32 bound = Chain::row_phase_bound(p.reserved);
                if (bound != 0u) {
                    bool outside = true;
#pragma unroll
                    for (int r = 0; r < ROWS; ++r) {
                        const int phase = W::row_phase(yw + r < ah ? yw + r : ah - 1, z, p.write) & int(bound);
                        seg[r] = int(block_x) * kRowsBX * V - (phase % x_group<R>() == 0 ? phase : 0);
                        whole = whole && seg[r] >= 0 && seg[r] + kRowsBX * V <= aw;
                        outside = outside && seg[r] >= aw;
                        x[r] = seg[r] + int(threadIdx.x) * V;
                    }
                    if (outside) return;                                   // (wave uniform, as `whole`)
                    if (whole) go(IntTag<0>{}); else go(IntTag<kRowEnds>{});
                    return;
                }
            }
#pragma unroll
            for (int r = 0; r < ROWS; ++r) { seg[r] = int(block_x) * kRowsBX * V; x[r] = seg[r] + int(threadIdx.x) * V; }
            whole = seg[0] + kRowsBX * V <= aw;
            if (whole) { go(IntTag<0>{}); return; }
            if (x[0] >= aw) return;
            go(IntTag<kRowEnd>{});
            return;
        }
    }
    const int x0 = (block_x * kRowsBX + threadIdx.x) * V;
    const int ybase = (block_y * kRowsBY + threadIdx.y) * ROWS;
    if (x0 >= aw || ybase >= ah) return;
    int same[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) same[r] = x0;
    if (!rows_any_x<Chain>(V) && x0 + V <= aw) {
        if constexpr (!rows_any_x<Chain>(V)) {
            if constexpr (kExchange) {
                if (int(block_x * kRowsBX + kRowsBX) * V <= aw) {
                    rows_full<Chain, V, ROWS, ALIGNED ? 2 : 2 | detail::kAnyAlign, kSmall>(p, kernarg_offset, same, same, ybase, z, aw, ah);
                    return;
                }
            }
            if constexpr (kMayStream) {
                if (stream) { rows_full<Chain, V, ROWS, (ALIGNED ? 1 : 0) | 4, false>(p, kernarg_offset, same, same, ybase, z, aw, ah); return; }
            }
            rows_full<Chain, V, ROWS, ALIGNED ? 1 : 0, kSmall>(p, kernarg_offset, same, same, ybase, z, aw, ah);
        }
    } else {
        for (int r = 0; r < ROWS; ++r) {
            const int y = ybase + r;
            if (y >= ah) break;
            for (int x = x0; x < aw; ++x) {
                Slot<typename R::Out> in[1];
                Slot<typename Chain::Value> out[1];
                in[0].v = R::exec(x, y, z, p.read);
                if constexpr (Chain::kLongChain) Chain::template compute_run_kernarg<1>(in, out, (const FKD_CONSTANT char*)__builtin_amdgcn_kernarg_segment_ptr() + kernarg_offset);
                else Chain::template compute_run<1>(in, out, p.ops);
                W::exec(x, y, z, out[0].v, p.write);
            }
        }
    }
}

// What one plane of a read is, and its parameters.
template <class R> struct ReadRoot { using Op = R; static constexpr bool batched = false; };
template <int N, class PlaneOp> struct ReadRoot<BatchRead<N, PlaneOp>> { using Op = PlaneOp; static constexpr bool batched = true; };

// ---- rows kernel, planes without gaps ----
//
// Images as decoders hand them over have no padding between their rows, so a plane is one row of w * h elements: segments of 256
// elements that begin where a line does follow each other through the whole plane, with no segment per row that is partly empty and no
// line that two waves share, and the kernel has no rows to work out.  A wave takes ROWS segments one after the other.  Bound by the memory
// (100 uchar3 images of 1527x794: 119 us for 728 MB) or, below 20 MB, by the launch and one trip to the memory.  us, rows / so:
// 4 uchar3 images of 1279x719 6.1 / 4.5, 100 of 103x243 7.9 / 4.0, of 439x918 55 / 41, of 1920x1080 208 / 204; floats 4 times 1861x714 through
// 30 operations 16.5 / 13.4, 4 of 317x63 through 100 20.6 / 11.9, 3840x2160 through 50 14.0 / 12.6.  Of 70 drawn sizes one got 1 % slower.
// The arguments that every wave needs are requested together and waited for once, and what is left of an address after the wave's own
// part is a lane's small offset.
template <class Chain> constexpr bool rows_flat() { return flat_capable<typename Chain::Read, typename Chain::Write>(); }
template <class Chain, int V, int ROWS, int MODE, bool PLAIN, bool EDGE, class Q, class WQ, class OPS>
__device__ __forceinline__ void flat_run(const Q& q, const WQ& wpar, const OPS& ops, int first, int total, int z) {
    using Op = typename ReadRoot<typename Chain::Read>::Op;
    using WP = typename Chain::Write::Plane;
    constexpr int kSegment = kRowsBX * V;
    const int lane = int(threadIdx.x);
    int x[ROWS], x0[ROWS];
    Slot<typename Op::Out> in[ROWS * V];
    // EDGE: some segment reaches past an end of the plane: lanes work on the first or last V elements instead and store the segment's own,
    // as in rows_full.
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        x0[r] = x[r] = (EDGE ? first : 0) + r * kSegment + lane * V;
        if constexpr (EDGE) x0[r] = x[r] < 0 ? 0 : (x[r] < total - V ? x[r] : total - V);
        Slot<typename Op::Out> row[V];
        Op::template exec_row<V, MODE>(x0[r], 0, z, q, row);
#pragma unroll
        for (int i = 0; i < V; ++i) in[r * V + i].v = row[i].v;
    }
    Slot<typename Chain::Value> out[ROWS * V];
    if constexpr (Chain::kLongChain) Chain::template compute_run_kernarg<ROWS * V>(in, out, (const FKD_CONSTANT char*)__builtin_amdgcn_kernarg_segment_ptr());
    else Chain::template compute_run<ROWS * V>(in, out, ops);
    constexpr int STORE = MODE | (PLAIN ? detail::kPlainStores : 0);
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        Slot<typename Chain::Value> row[V];
#pragma unroll
        for (int i = 0; i < V; ++i) row[i].v = out[r * V + i].v;
        if constexpr (!EDGE) {
            WP::template exec_row<V, STORE>(x0[r], 0, z, row, wpar);
        } else if constexpr (!PLAIN && has_edge_store<WP, V>()) {
            // (not in small launches, which are as long as their last wave: UYVY to float3 142x110 1.87 us without, 2.05 with it)
            if (first + r * kSegment < total) WP::template exec_edge<V>(first + r * kSegment, x0[r], total, 0, z, row, wpar);
        } else {
            if (x0[r] == x[r]) {
                WP::template exec_row<V, STORE>(x0[r], 0, z, row, wpar);
            } else if (x[r] > -V && x[r] < total) {
#pragma unroll
                for (int i = 0; i < V; ++i)
                    if (x0[r] + i >= x[r] && x0[r] + i < x[r] + V) WP::exec(x0[r] + i, 0, z, row[i].v, wpar);
            }
        }
    }
}
template <class Chain, int V, int ROWS, bool SMALL>
__device__ __forceinline__ void flat_body(const typename Chain::Params& p) {
    using Root = ReadRoot<typename Chain::Read>;
    using Op = typename Root::Op;
    using W = typename Chain::Write;
    using WP = typename W::Plane;
    static_assert(V == int(kFlatRun) && kRowsBX == 64 && kRowsBY == 4, "flat_blocks lays out the grid");
    constexpr int kSegment = kRowsBX * V;
    const int z = int(blockIdx.z);
    const typename Op::Params* rp;
    if constexpr (Root::batched) rp = &p.read.plane[z]; else rp = &p.read;
    typename Op::Params q = *rp;
    typename WP::Params wpar = W::plane_params(p.write, z);
    u32 head[4] = {p.active_w, p.active_h, p.reserved, gridDim.z};
    detail::pin_scalars(q);
    detail::pin_scalars(wpar);
    detail::pin_scalars(head);
    const int total = int(head[0] * head[1]);
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.y));
    int first = (int(blockIdx.x) * kRowsBY + wave) * ROWS * kSegment;
    if constexpr (!SMALL && has_row_phase<WP>()) {
        const int phase = WP::row_phase(0, z, wpar) & int(Chain::row_phase_bound(head[2]));
        first -= phase % x_group<Op>() == 0 ? phase : 0;
    }
    if (first >= total) return;
    constexpr bool kExchange = (detail::wave_exchange_ok<typename Op::Out>(V) || detail::wave_exchange_ok<typename W::In>(V));
    constexpr bool kMayStream = !SMALL && !Chain::kLongChain && !kExchange;
    constexpr int kWhole = kExchange ? 2 | detail::kAnyAlign : 0;
    if (first >= 0 && first + ROWS * kSegment <= total) {
        // the wave's own part as base addresses: what is left of an address is the lane's small offset
        Op::advance(q, first);
        WP::advance(wpar, first);
        if constexpr (kMayStream) {
            if ((unsigned long long)u32(total) * head[3] > kStreamElements) { flat_run<Chain, V, ROWS, kWhole | 4, SMALL, false>(q, wpar, p.ops, first, total, z); return; }
        }
        flat_run<Chain, V, ROWS, kWhole, SMALL, false>(q, wpar, p.ops, first, total, z);
    } else {
        flat_run<Chain, V, ROWS, 0, SMALL, true>(q, wpar, p.ops, first, total, z);
    }
}
template <class Chain, int V, int ROWS, bool SMALL>
__global__ __launch_bounds__(kRowsBX * kRowsBY) void k_flat(const typename Chain::Params p) {
    if constexpr (rows_flat<Chain>()) flat_body<Chain, V, ROWS, SMALL>(p);
}

// ---- rows kernel, scattered reads ----
//
// A warp's taps lie along a slanted line of the source, so what one instruction of a wave touches is decided by how far its
// lanes are apart in the output: with four adjacent outputs per lane, 64 lanes span 256 columns, which a turn by 7 degrees
// spreads over 31 source rows, nearly a cache line per lane and tap.  Here a wave owns 64 columns of the block's 256 and each
// lane one column of its four rows: an instruction spans 64 columns (8 rows at 7 degrees), its stores are 64 whole pixels
// side by side without an exchange through LDS, and what depends on the column serves four pixels.  What is left is bound by the
// lines the taps touch and the stores.  Four adjacent outputs per lane / one column of four rows, three sources and
// outputs in turn, us: 3840x2160 by 7 degrees 28.0 / 22.5, 2709x1462 by -18 degrees 19.8 / 14.5, perspective 1474x2063 by 29
// degrees 17.7 / 13.7, 4 of 811x319 13.9 / 12.1, 4 of 200x79 9.7 / 9.3.  (Lanes as 32 columns of two rows serve steep angles a little better,
// 13.1 for the 13.7, and everything else worse by 3 to 6 %: the stores' addresses are then the lanes' own.)
//
// The kernel's arguments are requested together and waited for once: a trip to the kernel-argument segment is 0.1 us of a
// launch of 2.3.
// For writers that store an element as one wide access; planar writers and elements of 1 to 3 bytes keep four outputs
// of a row per lane, which they store as one access.
template <class Op> constexpr bool reads_points() {
    if constexpr (requires { Op::kPoints; }) return Op::kPoints; else return false;
}
template <class Chain, int V, int ROWS> constexpr bool rows_by_points() {
    return V == kRowsBY && ROWS == 1 && reads_points<typename ReadRoot<typename Chain::Read>::Op>() && puts_whole<typename Chain::Write>();
}
template <class Chain, int V, int FORM>
__device__ __forceinline__ void points_body(const typename Chain::Params& p, const TileGeom& bands) {
    using Root = ReadRoot<typename Chain::Read>;
    using Op = typename Root::Op;
    using W = typename Chain::Write;
    using WP = typename W::Plane;
    constexpr bool kPhases = FORM == kRowsLines && has_row_phase<WP>();
    const int z = int(blockIdx.z);
    const typename Op::Params* rp;
    if constexpr (Root::batched) rp = &p.read.plane[z]; else rp = &p.read;
    TileGeom g = bands;
    typename Op::Params q = *rp;
    typename WP::Params wpar = W::plane_params(p.write, z);
    u32 head[3] = {p.active_w, p.active_h, p.reserved};
    detail::pin_scalars(g);
    detail::pin_scalars(q);
    detail::pin_scalars(wpar);
    detail::pin_scalars(head);
    const int aw = int(head[0]), ah = int(head[1]);
    u32 block_x = blockIdx.x, block_y = blockIdx.y;
    if (g.tiles_x != 0u) {
        // one band of the plane's blocks per XCD (see rows_in_bands); a two-dimensional grid holds exactly the plane's blocks
        const u32 gx = g.tiles_x, blocks = gx * g.tiles_y;
        u32 tin;
        if (g.n_tiles != 0u) {
            tin = (blockIdx.x % 8u) * rows_band_chunk(blocks) + blockIdx.x / 8u;
            if (tin >= blocks) return;
        } else {
            const u32 number = block_y * gx + block_x, k = number % 8u, rest = blocks % 8u;
            tin = k * (blocks / 8u) + (k < rest ? k : rest) + number / 8u;
        }
        block_y = g.tiles_x_magic ? u32(((unsigned long long)tin * g.tiles_x_magic) >> 32) : tin / gx;
        block_x = tin - block_y * gx;
    }
    const int lane = int(threadIdx.x), wave = __builtin_amdgcn_readfirstlane(int(threadIdx.y));
    const int left = int(block_x) * kRowsBX * V + wave * kRowsBX, top = int(block_y) * kRowsBY;
    u32 bound = 0;
    if constexpr (kPhases) bound = Chain::row_phase_bound(head[2]);
    if (left - int(bound) >= aw || top >= ah) return;
    int seg[V], x[V], y[V];
#pragma unroll
    for (int i = 0; i < V; ++i) { seg[i] = left; x[i] = left + lane; y[i] = top + i; }
    if constexpr (kPhases) {
        if (bound != 0u) {                              // (segments of 64 columns begin where a line does, see row_phase_bound)
#pragma unroll
            for (int i = 0; i < V; ++i) {
                seg[i] = left - (WP::row_phase(y[i] < ah ? y[i] : ah - 1, z, wpar) & int(bound));
                x[i] = seg[i] + lane;
            }
        }
    }
    Slot<typename Chain::Read::Out> in[V];
    Slot<typename Chain::Value> out[V];
    // (a second copy of the work for waves that are inside throughout costs launches of few waves more than it gives)
    Op::template exec_points<V, FORM == kRowsLines>(x, y, z, q, in, g.n_tiles != 0u);
    if constexpr (Chain::kLongChain) Chain::template compute_run_kernarg<V>(in, out, (const FKD_CONSTANT char*)__builtin_amdgcn_kernarg_segment_ptr());
    else Chain::template compute_run<V>(in, out, p.ops);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        typename WP::RowRef row = WP::row(y[i], z, wpar);
        row.p += seg[i];
        if (y[i] < ah && x[i] >= 0 && x[i] < aw) WP::template put<FORM == kRowsSmall>(row, lane, out[i].v);
    }
}

template <class Chain, int V, int ROWS, bool ALIGNED, int FORM>
__global__ __launch_bounds__(kRowsBX * kRowsBY) void k_rows(const typename Chain::Params p, const TileGeom g) {
    if constexpr (rows_by_points<Chain, V, ROWS>()) points_body<Chain, V, FORM>(p, g);
    else rows_body<Chain, V, ROWS, ALIGNED, rows_in_bands<Chain>(), FORM>(p, 0u, &g);
}

// Whether the rows of plane z of the read and of the write all start on dword boundaries, decided on the device
// (wave uniform, a handful of scalar instructions).  Kernels compiled at run time use this instead of the
// launcher's host-side check, because their launcher does not know the chain's type.
template <class Op, class P> FKD_DEV bool read_plane_aligned(const P& p, int z) {
    if constexpr (requires { Op::plane_rows_aligned(p, z, 0); }) return Op::plane_rows_aligned(p, z, 0);
    else return Op::rows_aligned(p, 0);
}
template <class Op, class P> FKD_DEV bool write_plane_aligned(const P& p, int z) {
    if constexpr (requires { Op::plane_rows_aligned(p, z); }) return Op::plane_rows_aligned(p, z);
    else return Op::rows_aligned(p);
}
template <class Chain, int V, int ROWS, bool BANDS = false, int FORM = kRowsOpen>
__device__ __forceinline__ void rows_auto_body(const typename Chain::Params& p, u32 kernarg_offset = 0, const TileGeom* bands = nullptr) {
    const int z = blockIdx.z;
    if constexpr (BANDS && rows_by_points<Chain, V, ROWS>()) { points_body<Chain, V, FORM>(p, *bands); return; }
    if constexpr (rows_any_x<Chain>(V)) { rows_body<Chain, V, ROWS, false, BANDS, FORM>(p, kernarg_offset, bands); return; }
    const bool aligned = read_plane_aligned<typename Chain::Read>(p.read, z) && write_plane_aligned<typename Chain::Write>(p.write, z);
    if (aligned) rows_body<Chain, V, ROWS, true, BANDS, FORM>(p, kernarg_offset, bands);
    else rows_body<Chain, V, ROWS, false, BANDS, FORM>(p, kernarg_offset, bands);
}

// ---- gather bilinear kernel ----------------------------------------------------------------------------

#ifndef FKD_GATHER_XI
#define FKD_GATHER_XI 2
#endif
#ifndef FKD_GATHER_YI
#define FKD_GATHER_YI 2
#endif
#ifndef FKD_GATHER_ADJ
#define FKD_GATHER_ADJ 0
#endif
#ifndef FKD_GATHER_BY
#define FKD_GATHER_BY 4
#endif
#ifndef FKD_GATHER_DEPTH
#define FKD_GATHER_DEPTH 2
#endif
constexpr int kGatherBX = 64;
constexpr int kGatherBY = FKD_GATHER_BY;

// A workgroup owns a (64*XI) x (4*YI) tile of the output of one plane; wave w owns rows w*YI .. w*YI+YI-1 of it, so
// everything that depends on the row (source rows, vertical weights, row addresses of source and destination) is
// wave uniform and lives in scalar registers.  A lane produces XI pixels (64 apart, so stores of a wave are
// contiguous) in each of its YI rows; the horizontal coordinate work is shared by the rows.  The four taps of a
// pixel are read straight from global memory as whole elements (a uchar3 comes in as one dword whose top byte is
// ignored); neighbouring lanes and rows hit the same cache lines, so HBM sees each source line about once.
// All loads of a lane are issued before the first use and are unconditional (coordinates are clamped into the
// source); only stores are predicated.
// The tile's work once the plane's parameters are in registers: q (the plane's read), ops, wpar (the plane's write), the
// output extent aw x ah, the plane z, the tile's first column tx0 and its row of tiles.
template <class Chain, int XI, int YI, bool STREAM, class Q, class OPS, class WPAR>
__device__ __forceinline__ void gather_tile(const typename Chain::Params& p, const Q& q, const OPS& ops, const WPAR& wpar,
                                            int aw, int ah, int z, int tx0, u32 tile_row) {
    using Root = ResizeRoot<typename Chain::Read>;
    using RZ = typename Root::Resize;
    using Back = typename RZ::BackOp;
    using Raw = typename Back::Raw;
    using W = typename Chain::Write;
    using WP = typename W::Plane;
    constexpr int TH = kGatherBY * YI;
    const int wy = __builtin_amdgcn_readfirstlane(int(threadIdx.y));
    const int y0 = int(tile_row) * TH + wy * YI;
    if (y0 >= ah) return;
    if constexpr (HasDefaultPlanes<typename Chain::Read>::value) {
        // BatchRead<CONDITIONAL_WITH_DEFAULT>: planes at or beyond `used` read nothing; every element is the default
        // value, which still goes through the chain's compute operations and the write.
        if (z >= p.read.used) {
            const typename RZ::Out def = p.read.def;
            const typename Chain::Value r = Chain::compute_checked_ops(def, ops);
            for (int y = y0; y < (y0 + YI < ah ? y0 + YI : ah); ++y) {
                const typename WP::RowRef orow = WP::row(y, z, wpar);
#pragma unroll
                for (int i = 0; i < XI; ++i) {
                    const int x = tx0 + int(threadIdx.x) + kGatherBX * i;
                    if (x < aw) WP::put(orow, x, r);
                }
            }
            return;
        }
    }
    int ox = 0, oy = 0;
    if constexpr (RZ::kAR != IGNORE_AR) { ox = q.x1; oy = q.y1; }
    const int sw = Back::width(q.back), sh = Back::height(q.back);

    // Pixels of a lane: XI adjacent ones (their results leave as one wide store per plane), or 64 apart.
    auto xof = [&](int i) {
        if constexpr (FKD_GATHER_ADJ) return tx0 + int(threadIdx.x) * XI + i;
        else return tx0 + int(threadIdx.x) + kGatherBX * i;
    };
    // Horizontal part, per lane, shared by the YI rows.  float(x1) and float(x1 + 1) are taken as floor(sx) and
    // floor(sx) + 1, the same numbers (exact integers below 2^24).
    int x1[XI], x2[XI];
    f32 ax[XI], bx[XI];
    bool xin[XI], clamped[XI];
    bool lane_clamped = false;
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        int x = xof(i);
        x = x < aw ? x : aw - 1;                                   // idle lanes shadow the last column
        xin[i] = true;
        if constexpr (RZ::kAR != IGNORE_AR) xin[i] = x >= q.x1 && x <= q.x2;
        const f32 sx = f32(x - ox) * q.fx;
        const f32 f1 = __builtin_floorf(sx);
        ax[i] = (f1 + 1.0f) - sx;
        bx[i] = sx - f1;
        const int xi = int(f1);
        x1[i] = xi < 0 ? 0 : (xi < sw - 1 ? xi : sw - 1);       // no-op wherever the reference is in bounds
        x2[i] = x1[i] + 1 < sw - 1 ? x1[i] + 1 : sw - 1;
        clamped[i] = x1[i] + 1 > sw - 1;
        lane_clamped = lane_clamped || clamped[i];
    }
    const bool any_clamped = __builtin_amdgcn_ballot_w64(lane_clamped) != 0;

    // Rows, software pipelined: the taps of row y+1 are requested before row y is blended, so once the first row
    // has arrived a wave always has data to work on while its next loads are in flight.  Two tap sets alternate
    // (the loop handles two rows per trip), so no registers are copied.
    // Three ways to fetch the taps of a row, chosen per wave:
    //   kPairs    the two horizontally adjacent taps of a pixel come in one access (possible when no lane of the
    //             wave has its right tap clamped to the last column), halving the number of gather instructions;
    //   kPairsSel the same for waves with clamped lanes: such a lane fetches the pair ending at the last column and
    //             uses its second element for both taps;
    //   kSingles  one access per tap, whole dwords;
    //   kSafe     one access per tap, never touching a byte outside the elements (channel by channel for 3- and
    //             6-byte elements): for waves whose taps reach the last row of the image.
    //   kPairsPrepared  kPairs for images whose rows all start at the same offset inside their dword (pitch a multiple
    //             of 4): the image is a buffer resource, a row a scalar offset, and the lane's window offset and byte
    //             shift are worked out once per column instead of once per tap;
    //   kWhole    both scale factors are whole numbers (4K -> 1080p): every source point is a pixel, the weights are
    //             1, 0, 0, 0, and the blend is the first tap; the others are not fetched.  Only for reads whose taps are
    //             always finite (a zero weight times them is a zero), and a lane whose first tap is a negative zero,
    //             where the zeros of the other three terms decide the sign of the sum, takes all four after all.
    constexpr int kSafe = 0, kSingles = 1, kPairs = 2, kPairsSel = 3, kPairsPrepared = 4, kWhole = 5;
    const int yend = y0 + YI < ah ? y0 + YI : ah;
    // STATIC: every quick operation of the chain takes its static form (decided once per wave, below).
    // Writers that can switch lanes off through their offset (kLaneMasked) store without an execution mask and with
    // 32-bit scalar row arithmetic; image planes too large for that (plane_maskable) take the plain stores.
    constexpr bool kCanMask = [] { if constexpr (requires { WP::kLaneMasked; }) return WP::kLaneMasked && !FKD_GATHER_ADJ; else return false; }();
    auto make_plane = [&] { if constexpr (kCanMask) return WP::plane_ref(z, wpar); else return 0; };
    const auto oplane = make_plane();
    u32 lane_off[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) { if constexpr (kCanMask) lane_off[i] = WP::lane_offset(xof(i), xof(i) < aw); else lane_off[i] = 0; }
    auto rows_with = [&](auto mode_tag, auto static_tag, auto masked_tag) {
        constexpr int MODE = decltype(mode_tag)::value;
        constexpr bool STATIC = decltype(static_tag)::value != 0;
        constexpr bool MASKED = decltype(masked_tag)::value != 0;
        constexpr bool PAIRED = MODE == kPairs || MODE == kPairsSel || MODE == kPairsPrepared;
        detail::PairPrep prep[XI];
        detail::TapImage image;
        if constexpr (MODE == kPairsPrepared) {
            image = Back::tap_image(z, q.back);
#pragma unroll
            for (int i = 0; i < XI; ++i) prep[i] = Back::pair_prepare(image, x1[i], q.back);
        }
        struct RowTaps {
            typename Back::TapBits a[PAIRED ? 1 : XI], b[PAIRED ? 1 : XI], c[PAIRED ? 1 : XI], d[PAIRED ? 1 : XI];
            typename Back::PairBits ab[PAIRED ? XI : 1], cd[PAIRED ? XI : 1];
            typename Back::TapRow ra, rb;
            f32 ay, by;
        };
        auto request = [&](int yrow, RowTaps& t) {
            const int y = yrow;
            const f32 sy = f32(y - oy) * q.fy;
            const f32 f1 = __builtin_floorf(sy);
            t.ay = (f1 + 1.0f) - sy;
            t.by = sy - f1;
            const int yi = __builtin_amdgcn_readfirstlane(int(f1));
            const int ya = yi < 0 ? 0 : (yi < sh - 1 ? yi : sh - 1);
            const int yb = ya + 1 < sh - 1 ? ya + 1 : sh - 1;
            if constexpr (MODE != kPairsPrepared) {
                t.ra = Back::tap_row(0, ya, z, q.back);
                t.rb = Back::tap_row(0, yb, z, q.back);
            } else {
                t.ra = typename Back::TapRow{};     // rows are scalar offsets into the image's buffer resource
                t.rb = typename Back::TapRow{};
            }
#pragma unroll
            for (int i = 0; i < XI; ++i) {
                if constexpr (MODE == kPairsPrepared) {
                    t.ab[i] = Back::pair_load_prepared(image, Back::tap_row_offset(ya, q.back), prep[i], q.back);
                    t.cd[i] = Back::pair_load_prepared(image, Back::tap_row_offset(yb, q.back), prep[i], q.back);
                } else if constexpr (PAIRED) {
                    const int xl = MODE == kPairsSel ? x1[i] - int(clamped[i]) : x1[i];
                    t.ab[i] = Back::pair_load(t.ra, xl, q.back);
                    t.cd[i] = Back::pair_load(t.rb, xl, q.back);
                } else if constexpr (MODE == kWhole) {
                    t.a[i] = Back::template tap_load<false>(t.ra, x1[i], q.back);
                } else {
                    t.a[i] = Back::template tap_load<MODE == kSingles>(t.ra, x1[i], q.back);
                    t.b[i] = Back::template tap_load<MODE == kSingles>(t.ra, x2[i], q.back);
                    t.c[i] = Back::template tap_load<MODE == kSingles>(t.rb, x1[i], q.back);
                    t.d[i] = Back::template tap_load<MODE == kSingles>(t.rb, x2[i], q.back);
                }
            }
        };
        auto produce = [&](int y, const RowTaps& t) {
            if (y >= yend) return;
            bool yin = true;
            if constexpr (RZ::kAR != IGNORE_AR) yin = y >= q.y1 && y <= q.y2;
            typename WP::RowRef orow;
            if constexpr (!MASKED) orow = WP::row(y, z, wpar);
            Slot<typename Chain::Value> res[XI];
#pragma unroll
            for (int i = 0; i < XI; ++i) {
                typename RZ::Taps tp;
                tp.w00 = ax[i] * t.ay; tp.w10 = bx[i] * t.ay; tp.w01 = ax[i] * t.by; tp.w11 = bx[i] * t.by;
                Raw a, b, c, d;
                if constexpr (MODE == kWhole) {
                    using Src = typename RZ::Src;
                    const Src first = Back::finish(Back::tap_value(t.a[i]), q.back);
                    typename RZ::Out v;
                    bool negative_zero = false;
                    auto take = [&](auto pa) {
                        const f32 f = f32(pa);
                        if constexpr (__is_same(base_t<Src>, f32) || __is_same(base_t<Src>, f64))
                            negative_zero = negative_zero || __builtin_bit_cast(u32, f) == 0x80000000u;
                        return f;
                    };
                    chan<0>(v) = take(chan<0>(first));
                    if constexpr (cn_v<Src> > 1) chan<1>(v) = take(chan<1>(first));
                    if constexpr (cn_v<Src> > 2) chan<2>(v) = take(chan<2>(first));
                    if constexpr (cn_v<Src> > 3) chan<3>(v) = take(chan<3>(first));
                    if (negative_zero) {
                        b = Back::tap_value(Back::template tap_load<false>(t.ra, x2[i], q.back));
                        c = Back::tap_value(Back::template tap_load<false>(t.rb, x1[i], q.back));
                        d = Back::tap_value(Back::template tap_load<false>(t.rb, x2[i], q.back));
                        v = RZ::blend(first, Back::finish(b, q.back), Back::finish(c, q.back), Back::finish(d, q.back), tp);
                    }
                    if constexpr (RZ::kAR != IGNORE_AR) { if (!(yin && xin[i])) v = q.bg; }
                    if constexpr (STATIC) res[i].v = Chain::compute_static_ops(v, ops);
                    else res[i].v = Chain::compute_checked_ops(v, ops);
                    continue;
                }
                if constexpr (PAIRED) {
                    const int xl = MODE == kPairsSel ? x1[i] - int(clamped[i]) : x1[i];
                    Back::pair_values(t.ab[i], t.ra, xl, a, b);
                    Back::pair_values(t.cd[i], t.rb, xl, c, d);
                    if constexpr (MODE == kPairsSel) { if (clamped[i]) { a = b; c = d; } }
                } else {
                    a = Back::tap_value(t.a[i]); b = Back::tap_value(t.b[i]);
                    c = Back::tap_value(t.c[i]); d = Back::tap_value(t.d[i]);
                }
                typename RZ::Out v = RZ::blend(Back::finish(a, q.back), Back::finish(b, q.back),
                                               Back::finish(c, q.back), Back::finish(d, q.back), tp);
                if constexpr (RZ::kAR != IGNORE_AR) { if (!(yin && xin[i])) v = q.bg; }
                if constexpr (STATIC) res[i].v = Chain::compute_static_ops(v, ops);
                else res[i].v = Chain::compute_checked_ops(v, ops);
            }
            if constexpr (MASKED) {
                const u32 row_off = masked_row_offset<WP>(y, oplane);
#pragma unroll
                for (int i = 0; i < XI; ++i) masked_put<WP, STREAM>(oplane, row_off, lane_off[i], res[i].v);
            } else if constexpr (FKD_GATHER_ADJ && XI > 1) {
                if (xof(XI - 1) < aw) {
                    WP::template put_run<XI>(orow, xof(0), res);
                } else {
#pragma unroll
                    for (int i = 0; i < XI; ++i) if (xof(i) < aw) WP::put(orow, xof(i), res[i].v);
                }
            } else {
#pragma unroll
                for (int i = 0; i < XI; ++i) if (xof(i) < aw) WP::put(orow, xof(i), res[i].v);
            }
        };
        if constexpr (YI == 1) {
            RowTaps t;
            request(y0, t);
            produce(y0, t);
        } else if constexpr (FKD_GATHER_DEPTH <= 2) {
            RowTaps t0, t1;
            request(y0, t0);
#pragma unroll 1
            for (int y = y0; y < yend; y += 2) {
                if (y + 1 < yend) request(y + 1, t1);      // wave uniform
                produce(y, t0);
                if (y + 2 < yend) request(y + 2, t0);
                produce(y + 1, t1);
            }
        } else {
            // A ring of DEPTH tap sets: DEPTH - 1 rows of loads stay in flight behind the row being blended.
            constexpr int D = FKD_GATHER_DEPTH;
            RowTaps t[D];
#pragma unroll
            for (int k = 0; k < D - 1; ++k) if (y0 + k < yend) request(y0 + k, t[k]);
#pragma unroll 1
            for (int y = y0; y < yend; y += D) {
#pragma unroll
                for (int k = 0; k < D; ++k) {
                    if (y + k + D - 1 < yend) request(y + k + D - 1, t[(k + D - 1) % D]);
                    produce(y + k, t[k]);
                }
            }
        }
    };
    auto rows = [&](auto mode_tag) {
        if constexpr (Chain::kQuick) {
            if (Chain::ops_static(ops)) { rows_with(mode_tag, IntTag<1>{}, IntTag<kCanMask ? 1 : 0>{}); return; }
        }
        rows_with(mode_tag, IntTag<0>{}, IntTag<kCanMask ? 1 : 0>{});
    };
    // Whole-dword reads of 3- and 6-byte elements (and pair reads) touch up to 3 bytes past what they need.  Inside
    // the image that is the next element or row; only in the image's last row it could leave the allocation.
    bool tail = false;
    if constexpr (Back::kTapOverread) {
        const int ylast = yend - 1;                                       // last row the wave requests
        const int yl = int(__builtin_floorf(f32(ylast - oy) * q.fy));
        const int yb = yl + 1 < sh - 1 ? yl + 1 : sh - 1;
        tail = Back::tap_last(Back::tap_row(0, yb < 0 ? 0 : yb, z, q.back));
    }
    if constexpr (kCanMask) {
        if (!WP::plane_maskable(wpar)) {
            if (tail) rows_with(IntTag<kSafe>{}, IntTag<0>{}, IntTag<0>{});
            else rows_with(IntTag<kSingles>{}, IntTag<0>{}, IntTag<0>{});
            return;
        }
    }
    if constexpr (finite_taps<Back>()) {
        // whole factors, and every source coordinate an exact float: decided on the host (ResizeLinear::whole_factors)
        if (q.whole) { rows(IntTag<kWhole>{}); return; }
    }
    if (tail) {
        rows(IntTag<kSafe>{});
    } else {
        if constexpr (Back::kTapPair) {
            if (!any_clamped) {
                if constexpr (detail::tap_prepared<Back>()) {
                    if (Back::tap_rows_share_alignment(q.back)) { rows(IntTag<kPairsPrepared>{}); return; }
                }
                rows(IntTag<kPairs>{});
                return;
            }
            if (sw >= 2) { rows(IntTag<kPairsSel>{}); return; }
        }
        rows(IntTag<kSingles>{});
    }
}

// Launches of few tiles.  A wave issues an instruction in four to five cycles at best, so where a SIMD has a wave or none the launch is as
// long as one wave's work: four pixels of 100 instructions are 0.8 us of a launch of 3.  Such launches take tiles of 64x4 pixels (one
// pixel per lane) or 128x4 (two); the line is at the number of 128x8 tiles the launch would have (gather_form, fkd/launch_info.hpp).
template <class Chain> constexpr u32 gather_some_tiles() {
    if constexpr (is_gather_chain<Chain>()) {
        if constexpr (requires { typename ResizeRoot<typename Chain::Read>::Resize::BackOp::FusedOver; }) return kGatherSomeTilesFused;
        else return kGatherSomeTiles;
    } else {
        return 0u;
    }
}

template <class Chain, int XI, int YI, bool STREAM>
__device__ __forceinline__ void gather_body(const typename Chain::Params& p, const TileGeom& g) {
    using Root = ResizeRoot<typename Chain::Read>;
    using RZ = typename Root::Resize;
    using W = typename Chain::Write;
    using WP = typename W::Plane;
    constexpr int TW = kGatherBX * XI;
    // The plane is the grid's z index, known at wave start, so the plane's parameters are fetched together with the
    // first kernel arguments instead of after them.  Within a plane workgroups are renumbered: hardware deals
    // consecutive workgroup ids round-robin to the 8 XCDs (the grid's x extent is a multiple of 8); XCD k gets the
    // k-th contiguous eighth of the plane's tiles so neighbouring tiles (which share source rows) share an L2.
    const int z = int(blockIdx.z);
    const typename RZ::Params* rp;
    if constexpr (Root::batched) rp = &p.read.plane[z]; else rp = &p.read;
    // A scalar load from the kernel-argument segment takes several hundred cycles, and a wave that lives for a few
    // thousand cannot afford one round trip per first use: geometry, the plane's read parameters, the operations'
    // parameters and the write's are requested back to back and waited for once.
    TileGeom gg = g;
    typename RZ::Params q = *rp;
    typename Chain::OpParams ops = p.ops;
    typename WP::Params wpar = W::plane_params(p.write, z);
    detail::pin_scalars(gg);
    detail::pin_scalars(q);
    detail::pin_scalars(ops);
    detail::pin_scalars(wpar);
    u32 dims[2] = {p.active_w, p.active_h};
    asm volatile("" : "+s"(dims[0]), "+s"(dims[1]));
    const int aw = int(dims[0]), ah = int(dims[1]);

    const u32 per_plane = gg.tiles_x * gg.tiles_y;
    const u32 chunk = (per_plane + 7u) / 8u;
    const u32 tin = (blockIdx.x % 8u) * chunk + blockIdx.x / 8u;
    if (tin >= per_plane) return;
    const u32 tile_row = gg.tiles_x_magic ? u32(((unsigned long long)tin * gg.tiles_x_magic) >> 32) : tin / gg.tiles_x;
    const int tx0 = int(tin - tile_row * gg.tiles_x) * TW;
    gather_tile<Chain, XI, YI, STREAM>(p, q, ops, wpar, aw, ah, z, tx0, tile_row);
}

// ---- strip form of the bilinear kernel: narrow outputs (batches of small planes) -------------------------------------
//
// A workgroup of four waves owns 8 whole output rows of one plane, up to 256 pixels wide.  A HALF wave (32 lanes) owns
// one row and each lane the columns lane, lane + 32, lane + 64, ...: a 224-pixel row is seven such steps with no idle
// lane, where 128-pixel tiles leave one lane in eight without work.  What depends on the column (horizontal weights,
// the byte offset of the tap window and the bytes to drop from it) is worked out ONCE per workgroup, one column per
// thread, and handed round through 4 KB of LDS; what depends on the row is worked out once per lane and serves all its
// pixels.  So the fixed work of a wave is spread over seven pixels per lane instead of four, nearly all of it on the
// vector unit (the scalar unit is shared by the four SIMDs of a compute unit and was as busy as they were).
// What the form asks of every plane -- source smaller than 2 GB and at least two columns wide, output plane smaller than 2 GB -- is checked on the host when the parameter
// block is made (Chain::finalize_write, bit 0 of Params::reserved); launchers take the tile form when the bit is clear.
// Taps come through a buffer resource whose extent ends with the image, so windows that reach past the last row read
// zeros in bytes nobody uses and no lane needs a narrower access; the row is part of the lane's offset.
// Wave priorities of the strip form.  A SIMD serves its oldest wave first, so in a launch that fits the chip in one round
// (every workgroup resident from the start: configuration 3's 1 792) the seven waves of a SIMD do not advance side by side:
// the wave that was started last is held back at every stage and ends up walking its steps nearly alone, each step exposed
// to the full latency of its taps (measured with per-wave time stamps: the first wave of a SIMD issues its last stores 3.6 us
// after the launch's first wave entered, the seventh 7.5 us).  Such a launch therefore starts every wave at priority 3 and
// lowers it as the wave advances (2 from step 3, 1 from step 5), which makes the waves of a SIMD advance together; and
// workgroups that were started late (the dispatcher hands consecutive workgroup numbers round the compute units, so a
// workgroup's number divided by the number of compute units says roughly how many were on its unit before it) keep each
// level one step longer, which is what keeps the last wave of a SIMD from finishing alone.  Configuration 3: 8.15 -> 7.85 us.
// A launch of several rounds is left alone: the fresh waves of a later round would outrank the last steps of the round
// before (twice the rows: 14.1 -> 15.4 us with the priorities on).  Priorities change the order of issue, never a result.
// The launcher decides and hands the kernel one number: the number of the first workgroup that counts as started late, or
// 0 for a launch whose waves keep the default priority.
// (strip_first_late_workgroup, fkd/launch_info.hpp)
constexpr int kStripRows = int(kStripFormRows), kStripStep = 32, kStripMaxWidth = 256;
constexpr int kStripThreads = kStripRows * kStripStep, kStripMaxSteps = kStripMaxWidth / kStripStep;
static_assert(kStripThreads == kGatherBX * kGatherBY, "the two forms of the bilinear kernel share their workgroup shape");
static_assert(kStripThreads == kStripMaxWidth, "one table column per thread");

template <class Chain> constexpr bool strip_capable() {
    using Root = ResizeRoot<typename Chain::Read>;
    if constexpr (!Root::value) return false;
    else if constexpr (HasDefaultPlanes<typename Chain::Read>::value) return false;
    else {
        using Back = typename Root::Resize::BackOp;
        using WP = typename Chain::Write::Plane;
        if constexpr (!detail::tap_prepared<Back>()) return false;
        else if constexpr (!Back::kTapPair) return false;
        else if constexpr (requires { WP::kLaneMasked; }) return WP::kLaneMasked;
        else return false;
    }
}

// Planar outputs whose rows are no whole lines: the stores of a row's steps, moved on to line boundaries.
//
// A step's LANES values begin wherever the row does, so stored as they are they cut a line at both of their ends, and such a line
// leaves the chip as two partial writes (64 crops to 639x639 104 us where 640x640 take 57).  Here the lanes of a step store the
// LANES elements from a line boundary on: a lane takes its value from the lane `shift` below it (ds_bpermute), and the lanes below the shift
// store what the step before has left.  Channel planes begin anywhere too, so each has a shift of its own.  Only the two lines at a row's ends
// are cut.  (Whole strips collected in LDS and stored as one run cut fewer lines and were slower for all but the largest launches: 225x225
// 13.0 against 11.5 us, 517x517 52.5 / 48.2, 639x639 75 / 81; the LDS leaves room for three or four workgroups, and stores begin when a
// workgroup's work is over.)
template <class Chain, int LANES> struct LineStores {
    using Value = typename Chain::Value;
    using WP = typename Chain::Write::Plane;
    static constexpr int N = cn_v<Value>;
    u32 off[N];        // byte offset of the lane's element of step 0
    int from[N];       // the lane (times four) whose value the lane stores
    int shift[N];      // elements between the line boundary at or before the row's first element and that element
    u32 left[N];       // what the step before left for the lanes below the shift
    // g: the lane's number in its row
    template <class WPAR> __device__ __forceinline__ void open(int z, int y, bool valid, int g, const WPAR& wpar) {
        const char* row = WP::channel_row(z, y, wpar);
        const u32 row_off = u32(row - WP::channel_row(z, 0, wpar));
        const int lane0 = int(threadIdx.x) - g;
#pragma unroll
        for (int c = 0; c < N; ++c) {
            shift[c] = int((u32(reinterpret_cast<uintptr_t>(row + size_t(c) * WP::channel_bytes(wpar))) / 4u) & (kLineBytes / 4u - 1u));
            off[c] = valid ? row_off + u32(g - shift[c]) * 4u : WP::kMaskedOut;
            from[c] = (lane0 + ((g - shift[c]) & (LANES - 1))) * 4;
            left[c] = 0u;
        }
    }
    // (the offset of a lane left of its row wraps, but such a lane is masked: check)
    template <bool STREAM, int C> __device__ __forceinline__ void store(const typename WP::PlaneRef& r, int k, int g, bool check, int aw, u32 now) {
        const u32 v = g < shift[C] ? left[C] : now;
        u32 at = off[C] + u32(k) * (LANES * 4u);
        if (check) {
            const int x = k * LANES + g - shift[C];
            if (x < 0 || x >= aw) at = WP::kMaskedOut;
        }
        WP::template put_channel<STREAM, C>(r, at, v);
        left[C] = now;
    }
    template <bool STREAM, int C> __device__ __forceinline__ void one(const typename WP::PlaneRef& r, int k, int g, bool check, int aw, const Value& v) {
        store<STREAM, C>(r, k, g, check, aw, u32(__builtin_amdgcn_ds_bpermute(from[C], int(__builtin_bit_cast(u32, chan<C>(v))))));
    }
    template <bool STREAM> __device__ __forceinline__ void put(const typename WP::PlaneRef& r, int k, int g, bool check, int aw, const Value& v) {
        one<STREAM, 0>(r, k, g, check, aw, v); one<STREAM, 1>(r, k, g, check, aw, v);
        if constexpr (N > 2) one<STREAM, 2>(r, k, g, check, aw, v);
        if constexpr (N > 3) one<STREAM, 3>(r, k, g, check, aw, v);
    }
    // ... and what the last step left.
    template <bool STREAM> __device__ __forceinline__ void finish(const typename WP::PlaneRef& r, int steps, int g, int aw) {
        store<STREAM, 0>(r, steps, g, true, aw, 0u); store<STREAM, 1>(r, steps, g, true, aw, 0u);
        if constexpr (N > 2) store<STREAM, 2>(r, steps, g, true, aw, 0u);
        if constexpr (N > 3) store<STREAM, 3>(r, steps, g, true, aw, 0u);
    }
};

// ANY_PITCH: some image of the launch has rows that do not share their alignment (Chain::kStripAnyPitch).
// LINES: stores on line boundaries (LineStores); then a row may have LANES = 64 lanes, so a workgroup four rows, and MAX_STEPS steps.
template <class Chain, bool STREAM, bool ANY_PITCH, bool LINES = false, int LANES = kStripStep, int MAX_STEPS = kStripMaxSteps>
__device__ __forceinline__ void strip_body(const typename Chain::Params& p, const u32 first_late_workgroup) {
    constexpr int kStripStep = LANES, kStripMaxSteps = MAX_STEPS, kStripRows = kStripThreads / LANES;
    constexpr int kColumns = LINES ? (MAX_STEPS + 1) * LANES : kStripMaxWidth;
    using Root = ResizeRoot<typename Chain::Read>;
    using RZ = typename Root::Resize;
    using Back = typename RZ::BackOp;
    using Raw = typename Back::Raw;
    using W = typename Chain::Write;
    using WP = typename W::Plane;
    // per column: ax, bx, window offset, bytes to drop from the window (bits 0-1) | flags
    __shared__ detail::u32x4_t column[kColumns];
    __shared__ u32 wave_clamped[kStripThreads / 64];
    constexpr u32 kClamped = 0x80000000u, kOutsideX = 0x40000000u;

    const int z = int(blockIdx.z);
    // every wave starts at the highest priority, before its arguments are there: a launch of more than one round drops
    // it again below, once they say so
    __builtin_amdgcn_s_setprio(3);
    const typename RZ::Params* rp;
    if constexpr (Root::batched) rp = &p.read.plane[z]; else rp = &p.read;
    typename RZ::Params q = *rp;
    typename Chain::OpParams ops = p.ops;
    typename WP::Params wpar = W::plane_params(p.write, z);
    u32 dims[4] = {p.active_w, p.active_h, first_late_workgroup, gridDim.x};
    detail::pin_scalars(q);
    detail::pin_scalars(ops);
    detail::pin_scalars(wpar);
    // (the grid's width with the rest: fetched where it is used, it would be a second trip to the kernel-argument segment)
    asm volatile("" : "+s"(dims[0]), "+s"(dims[1]), "+s"(dims[2]), "+s"(dims[3]));
    const int aw = int(dims[0]), ah = int(dims[1]);
    // the steps at which this wave's priority falls to 2 and to 1, as two scalars (wave uniform)
    int falls[2] = {3, 5};
    if (dims[2] == 0u) {
        __builtin_amdgcn_s_setprio(0);
        falls[0] = falls[1] = kStripMaxSteps;                           // never
    } else if (blockIdx.z * dims[3] + blockIdx.x >= dims[2]) {
        falls[0] = 4;
        falls[1] = 6;
    }
    asm volatile("" : "+s"(falls[0]), "+s"(falls[1]));
    int ox = 0, oy = 0;
    if constexpr (RZ::kAR != IGNORE_AR) { ox = q.x1; oy = q.y1; }
    const int sw = Back::width(q.back), sh = Back::height(q.back);
    const detail::TapImage image = Back::tap_image_bounded(z, q.back);
    // Rows that do not share their alignment: a column's entry then holds the byte offset of its first tap, and where in its
    // dword the window begins is only known together with the row (one more instruction per pixel and line).  Otherwise it
    // holds the offset of the window.  For pixels of whole dwords the two are the same: their windows begin with the first tap,
    // whatever its address.
    using Window = typename Back::PairBits;
    // Each kind has a kernel of its own: with both in one, its code half as long again, launches of more than one workgroup per
    // compute unit were 2 to 7 % slower, of either kind (8 crops to 128x640 3.31 -> 3.51 us).
    constexpr bool kAnyPitch = Window::kShift && ANY_PITCH;
    const int steps = (aw + kStripStep - 1) / kStripStep;
    if (steps == 0) return;                                             // no columns: nothing to write (the whole workgroup leaves)
    // With lines the launches are larger, and one whose planes are tall or share their source (large crops of one image) would have every XCD
    // fetch all of it; as bands, us, without / with / the forms that such launches took before there were line stores: 8 crops of 1200x800 to 225x500
    // 7.05 / 4.70 / 5.26, to 255x1000 9.4 / 6.9 / 7.4, to 331x331 6.88 / 4.90 / 5.15, to 435x435 8.6 / 6.4 / 6.6; one image of 1200x800, compiled
    // at run time: ushort3 to 255x12001 16.7 / 10.7 / 10.6, to 333x4003 7.53 / 5.9 / 6.3, uchar4 to 129x6001 7.1 / 5.6 / 6.1.  Launches of a few
    // microseconds pay 0.05 to 0.1 us for it (64 crops to 258x40 4.40 / 4.49 / 5.05, 8 to 299x299 4.39 / 4.55 / 5.0).
    const u32 strip = LINES ? plane_band(blockIdx.x, dims[3], blockIdx.z) : blockIdx.x;

    const int t = int(threadIdx.y) * 64 + int(threadIdx.x);
    // What depends on the column: the horizontal weights, the window's byte offset in a row, and flags beside the bytes to drop.
    auto column_entry = [&](int col, bool& clamped) {
        const int x = col < aw ? col : aw - 1;                          // columns beyond the output shadow the last one
        const f32 sx = f32(x - ox) * q.fx;
        const f32 f1 = __builtin_floorf(sx);
        const f32 ax = (f1 + 1.0f) - sx, bx = sx - f1;
        const int xi = int(f1);
        const int x1 = xi < 0 ? 0 : (xi < sw - 1 ? xi : sw - 1);
        clamped = x1 + 1 > sw - 1;                                      // right tap is the last column again
        const detail::PairPrep pp = Back::pair_prepare(image, x1 - int(clamped), q.back);
        u32 flags = pp.shift | (clamped ? kClamped : 0u);
        if constexpr (RZ::kAR != IGNORE_AR) flags |= (x >= q.x1 && x <= q.x2) ? 0u : kOutsideX;
        detail::u32x4_t e;
        e.x = __builtin_bit_cast(u32, ax); e.y = __builtin_bit_cast(u32, bx); e.z = kAnyPitch ? pp.off + pp.shift : pp.off; e.w = flags;
        return e;
    };

    // ---- the lane's row ----
    const int g = t & (kStripStep - 1), r = t / kStripStep;
    const int y = int(strip) * kStripRows + r;
    const bool yvalid = y < ah;
    const int yc = yvalid ? y : ah - 1;
    const f32 sy = f32(yc - oy) * q.fy;
    const f32 fy1 = __builtin_floorf(sy);
    const f32 ay = (fy1 + 1.0f) - sy, by = sy - fy1;
    const int yi = int(fy1);
    const int ya = yi < 0 ? 0 : (yi < sh - 1 ? yi : sh - 1);
    const int yb = ya + 1 < sh - 1 ? ya + 1 : sh - 1;
    const u32 row_a = Back::tap_row_offset(ya, q.back), row_b = Back::tap_row_offset(yb, q.back);
    bool yin = true;
    if constexpr (RZ::kAR != IGNORE_AR) yin = yc >= q.y1 && yc <= q.y2;

    struct StepTaps { detail::u32x4_t e; typename Back::PairBits ab, cd; };
    auto fetch = [&](StepTaps& s) {
        // (v_alignbyte_b32 takes the bytes to drop from bits 0-1 of its operand, so the flags may ride along)
        detail::PairPrep pa, pb;
        pa.off = s.e.z + row_a; pa.shift = s.e.w;
        pb.off = s.e.z + row_b; pb.shift = s.e.w;
        if constexpr (kAnyPitch) {
            pa = detail::pair_window_at<Window>(pa.off);
            pb = detail::pair_window_at<Window>(pb.off);
        }
        s.ab = Back::pair_load_prepared(image, 0u, pa, q.back);
        s.cd = Back::pair_load_prepared(image, 0u, pb, q.back);
    };
    auto request = [&](int k, StepTaps& s) {
        s.e = column[g + kStripStep * k];
        fetch(s);
        __builtin_amdgcn_sched_barrier(0);      // the next step's taps leave before anything waits for this step's
    };
    // The taps of step 0 are requested before the table exists, from the lane's own working out of its first column:
    // they are then on their way while the table is made and the workgroup meets at the barrier.
    StepTaps first;
    {
        bool unused;
        first.e = column_entry(g, unused);
        fetch(first);
    }

    // ---- the column table: one column per thread (the workgroup has as many threads as the form has columns).  Columns
    // of the steps after the last one hold a window offset of 2 GB: the image is smaller than that (checked on the host), so
    // the sum with the lane's row offset neither wraps nor comes back below the image's extent, and requesting such a
    // column touches no memory.  Each wave notes whether it met a clamped column. ----
    constexpr u32 kNoWindow = 0x80000000u;
    {
        bool clamped = false;
        if constexpr (LINES) {
            // (up to a step behind the last one, which the request behind the last step meets)
            for (int c = t; c < (steps + 1) * kStripStep; c += kStripThreads) {
                detail::u32x4_t e = column_entry(c, clamped);
                if (c >= steps * kStripStep) e.z = kNoWindow;
                column[c] = e;
            }
        } else {
            detail::u32x4_t e = column_entry(t, clamped);
            if (t >= steps * kStripStep) { e.z = kNoWindow; clamped = false; }
            column[t] = e;
        }
        const bool any = __builtin_amdgcn_ballot_w64(clamped) != 0ull;
        if (threadIdx.x == 0) wave_clamped[threadIdx.y] = any ? 1u : 0u;
    }
    __syncthreads();
    u32 met = 0;
#pragma unroll
    for (int w = 0; w < kStripThreads / 64; ++w) met |= wave_clamped[w];
    const bool some_clamped = __builtin_amdgcn_readfirstlane(met) != 0u;

    const auto oplane = WP::plane_ref(z, wpar);
    LineStores<Chain, LANES> lines;
    if constexpr (LINES) lines.open(z, yc, yvalid, g, wpar);
    // the lane's store offset in step 0; a lane without a row carries an offset beyond the resource's extent
    const u32 out0 = yvalid ? WP::row_offset(y, oplane) + WP::lane_offset(g, true) : WP::kMaskedOut;
    const bool partial = (aw & (kStripStep - 1)) != 0;             // the last step has columns beyond the output

    auto run = [&](auto static_tag, auto clamp_tag) {
        constexpr bool STATIC = decltype(static_tag)::value != 0;
        constexpr bool CLAMP = decltype(clamp_tag)::value != 0;
        auto produce = [&](int k, const StepTaps& s) {
            // (k is known where the steps are written out: one comparison in four of the steps)
            if ((k == 3 || k == 4) && k == falls[0]) __builtin_amdgcn_s_setprio(2);
            if ((k == 5 || k == 6) && k == falls[1]) __builtin_amdgcn_s_setprio(1);
            // (the words are copied out first: a bit cast applied directly to an element of the vector reads element 0)
            const u32 ax_bits = s.e.x, bx_bits = s.e.y;
            const f32 ax = __builtin_bit_cast(f32, ax_bits), bx = __builtin_bit_cast(f32, bx_bits);
            typename RZ::Taps tp;
            tp.w00 = ax * ay; tp.w10 = bx * ay; tp.w01 = ax * by; tp.w11 = bx * by;
            Raw a, b, c, d;
            if constexpr (CLAMP) {
                const bool clamped = (s.e.w & kClamped) != 0u;
                Back::pair_values_dup(s.ab, clamped, a, b);
                Back::pair_values_dup(s.cd, clamped, c, d);
            } else {
                Back::pair_values(s.ab, typename Back::TapRow{}, 0, a, b);
                Back::pair_values(s.cd, typename Back::TapRow{}, 0, c, d);
            }
            typename RZ::Out v = RZ::blend(Back::finish(a, q.back), Back::finish(b, q.back),
                                           Back::finish(c, q.back), Back::finish(d, q.back), tp);
            if constexpr (RZ::kAR != IGNORE_AR) { if (!yin || (s.e.w & kOutsideX)) v = q.bg; }
            typename Chain::Value res;
            if constexpr (STATIC) res = Chain::compute_static_ops(v, ops);
            else res = Chain::compute_checked_ops(v, ops);
            if constexpr (LINES) { lines.template put<STREAM>(oplane, k, g, k == 0 || k == steps - 1, aw, res); return; }
            u32 off = out0 + u32(k) * WP::lane_offset(kStripStep, true);
            if (partial && k == steps - 1) {                          // wave uniform, kept a branch
                asm volatile("" : "+v"(off));
                if (g + kStripStep * k >= aw) off = WP::kMaskedOut;
            }
            WP::template put_masked<STREAM>(oplane, 0u, off, res);
        };
        // One step of taps is in flight behind the step being blended.  The steps are written out (a plane has at most
        // kStripMaxSteps of them) and the only branches leave them (for good, or with LINES for finish, which stores what is left): every step issues the same accesses in the same
        // order, so the compiler's wait for a step's taps leaves all later accesses in flight, table reads carry their step
        // in the instruction's immediate offset, and there is no loop bookkeeping.  The request behind the last step meets
        // a column without a window.
        StepTaps sa = first, sb;
        request(1, sb);
#pragma unroll
        for (int k = 0; k < kStripMaxSteps; k += 2) {
            if (k > 0) request(k + 1, sb);
            produce(k, sa);
            if (k + 1 >= steps) return;
            if (k + 2 < kStripMaxSteps) request(k + 2, sa);
            produce(k + 1, sb);
            if (k + 2 >= steps) return;
        }
    };
    auto run_static = [&](auto static_tag) {
        if (kAnyPitch || some_clamped) run(static_tag, IntTag<1>{});
        else run(static_tag, IntTag<0>{});
    };
    auto finish = [&] { if constexpr (LINES) lines.template finish<STREAM>(oplane, steps, g, aw); };
    if constexpr (Chain::kQuick) {
        if (Chain::ops_static(ops)) { run_static(IntTag<1>{}); finish(); return; }
    }
    run_static(IntTag<0>{});
    finish();
}

// (both kinds of image rows in one kernel: the instruction more per pixel and line is nothing beside the stores)
template <class Chain, bool STREAM, int LANES>
__device__ __forceinline__ void strip_lines_body(const typename Chain::Params& p) {
    strip_body<Chain, STREAM, true, true, LANES, LANES == 32 ? kStripMaxSteps : int(kLinesWidth) / 64>(p, 0u);
}
template <class Chain, bool STREAM, int LANES>
__global__ __launch_bounds__(kStripThreads) void k_strip_lines(const typename Chain::Params p) {
    if constexpr (strip_capable<Chain>()) strip_lines_body<Chain, STREAM, LANES>(p);
}

template <class Chain, bool STREAM, bool ANY_PITCH>
__global__ __launch_bounds__(kStripThreads) void k_strip(const typename Chain::Params p, const u32 first_late_workgroup) {
    if constexpr (strip_capable<Chain>()) strip_body<Chain, STREAM, ANY_PITCH>(p, first_late_workgroup);
}

template <class Chain, int XI, int YI, bool STREAM>
__global__ __launch_bounds__(kGatherBX * kGatherBY) void k_gather(const typename Chain::Params p, const TileGeom g) {
    gather_body<Chain, XI, YI, STREAM>(p, g);
}

// ---- per-chain constants shared by the ahead-of-time and the run-time launchers ---------------------------

template <class Chain> struct RowsConfig {
    // Four elements per thread; a bilinear resize without a tap cursor keeps one element per thread.  (Warps take four
    // as well, of one column: points_body.)
    static constexpr bool kScattered = ResizeRoot<typename Chain::Read>::value;
#ifndef FKD_ROWS
#define FKD_ROWS 2
#endif
#ifndef FKD_SCATTER_V
#define FKD_SCATTER_V 1
#endif
#ifndef FKD_SCATTER_ROWS
#define FKD_SCATTER_ROWS 1
#endif
    static constexpr int V = kScattered ? FKD_SCATTER_V : 4;
    // Two rows per thread; chains long enough to be bound by instruction issue rather than by memory (more than 128
    // bytes of operation parameters) take four, for the independent work per thread.
    static constexpr bool kManyOps = sizeof(typename Chain::Params) - sizeof(typename Chain::Read::Params) - sizeof(typename Chain::Write::Params) > 128 + 16;
#ifndef FKD_ROWS_MANY
#define FKD_ROWS_MANY (2 * FKD_ROWS)
#endif
    static constexpr int ROWS = (kScattered || is_scattered_read<typename Chain::Read>()) ? FKD_SCATTER_ROWS : (kManyOps ? FKD_ROWS_MANY : FKD_ROWS);
};

// Below how many workgroups a launch takes half the rows per thread (see kRowsFewBlocks).
template <class Chain> constexpr u32 rows_few_blocks() {
    constexpr int V = RowsConfig<Chain>::V;
    return detail::wave_exchange_ok<typename Chain::Read::Out>(V) || detail::wave_exchange_ok<typename Chain::Write::In>(V) ? kRowsFewBlocksExchange : kRowsFewBlocks;
}

// Chains that keep all their rows in launches of kRowsWholeFrom to kRowsWholeTo workgroups: reads of two-plane video, and images whose elements are
// exchanged between the lanes where they are read and where they are written.
template <class Op> constexpr bool reads_two_planes() {
    if constexpr (requires { typename Op::FusedOver; }) return reads_two_planes<typename Op::FusedOver>();
    else if constexpr (requires { Op::kTwoPlanes; }) return Op::kTwoPlanes;
    else return false;
}
template <class Op> constexpr bool reads_exchanged(int v) {
    if constexpr (requires { typename Op::FusedOver; }) return reads_exchanged<typename Op::FusedOver>(v);
    else return knows_dense<Op>() && detail::wave_exchange_ok<typename Op::Out>(v);
}
template <class Chain> constexpr bool rows_keep_whole() {
    using Op = typename ReadRoot<typename Chain::Read>::Op;
    constexpr int V = RowsConfig<Chain>::V;
    return reads_two_planes<Op>() || (reads_exchanged<Op>(V) && detail::wave_exchange_ok<typename Chain::Write::In>(V) && puts_whole<typename Chain::Write>());
}

// ---- divergent batch kernel -------------------------------------------------------------------------------

// Several chains in one launch of the rows kernel's geometry: plane z runs chain select[z] (wave uniform: the plane is
// the grid's z index).  Every chain runs through the rows body, bilinear reads included, all with the same elements per
// thread; workgroups beyond a chain's own extent leave at once.
template <class... Chains> struct RowsConfig<Divergent<Chains...>> {
    // One geometry for every chain of the launch, gathering reads included (they then take their elements one after
    // the other): with the grid laid out for the finest chain, the planes of the coarser ones launched up to 16 times
    // the workgroups they needed, and those empty workgroups cost 4 us of a 31 us launch.
    static constexpr int V = 4;
    static constexpr int ROWS = FKD_ROWS;
};
template <int I, class First, class... Rest, class P>
__device__ __forceinline__ void divergent_run(u32 sel, const P& p, const Tup<typename First::Params, typename Rest::Params...>& seq) {
    if (sel == u32(I)) {
        const u32 offset = u32(reinterpret_cast<const char*>(&seq.head) - reinterpret_cast<const char*>(&p));
        rows_auto_body<First, 4, FKD_ROWS>(seq.head, offset);
    } else if constexpr (sizeof...(Rest) > 0) {
        divergent_run<I + 1, Rest...>(sel, p, seq.tail);
    }
}
template <class D> struct DivergentBody;
template <class... Chains> struct DivergentBody<Divergent<Chains...>> {
    __device__ __forceinline__ static void run(const typename Divergent<Chains...>::Params& p) {
        using D = Divergent<Chains...>;
        const u32 z = blockIdx.z < u32(D::kMaxPlanes) ? blockIdx.z : 0u;
        // The table entry is fetched from the kernel-argument segment itself (the parameter block is the kernel's first
        // argument): indexing the by-value copy with a run-time index would make the compiler keep that copy in
        // scratch memory, for every lane.
        const FKD_CONSTANT u32* words = (const FKD_CONSTANT u32*)__builtin_amdgcn_kernarg_segment_ptr();
        const u32 at = u32(__builtin_offsetof(typename D::Params, select)) + z;
        const u32 sel = __builtin_amdgcn_readfirstlane((words[at / 4u] >> ((at & 3u) * 8u)) & 0xffu);
        divergent_run<0, Chains...>(sel, p, p.seq);
    }
};
template <class D> __global__ __launch_bounds__(kRowsBX * kRowsBY) void k_divergent(const typename D::Params p) {
    DivergentBody<D>::run(p);
}

// The one kernel of a chain compiled at run time, and what its launcher needs to know about it.  A launcher that
// only has the parameter block as bytes reads the active grid from its first three words.
// Whether the chain has a kernel for small outputs.
template <class Chain> constexpr bool rows_have_small() {
    if constexpr (IsDivergent<Chain>::value) return false; else return !is_gather_chain<Chain>();
}
// ... and kernels for planes without gaps.
template <class Chain> constexpr bool rows_have_flat() {
    if constexpr (IsDivergent<Chain>::value) return false; else return !is_gather_chain<Chain>() && rows_flat<Chain>();
}
// (JitMeta: fkd/launch_info.hpp)
template <class Chain> constexpr JitMeta jit_meta() {
    if constexpr (IsDivergent<Chain>::value)
        return JitMeta{0u, u32(sizeof(typename Chain::Params)), u32(RowsConfig<Chain>::V), u32(RowsConfig<Chain>::ROWS), 0u, 0u, 0u, u32(Chain::kMaxPlanes), 0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    else
        return JitMeta{is_gather_chain<Chain>() ? 1u : 0u, u32(sizeof(typename Chain::Params)), u32(RowsConfig<Chain>::V),
                       u32(RowsConfig<Chain>::ROWS), u32(FKD_GATHER_XI), u32(FKD_GATHER_YI), u32(kGatherBY), 0u,
                       is_gather_chain<Chain>() && strip_capable<Chain>() ? u32(kStripMaxWidth) : 0u,
                       !is_gather_chain<Chain>() && rows_in_bands<Chain>() ? (rows_by_points<Chain, RowsConfig<Chain>::V, RowsConfig<Chain>::ROWS>() ? 2u : 1u) : 0u, rows_have_small<Chain>() ? 1u : 0u, rows_have_flat<Chain>() ? 1u : 0u,
                       is_gather_chain<Chain>() && writer_streams<Chain>() ? u32(sizeof(typename Chain::Value)) : 0u,
                       gather_some_tiles<Chain>(), rows_few_blocks<Chain>(), rows_keep_whole<Chain>() ? 1u : 0u};
}
template <class Chain> __device__ __forceinline__ void jit_body(const typename Chain::Params& p, const TileGeom& g) {
    if constexpr (IsDivergent<Chain>::value) DivergentBody<Chain>::run(p);
    else if constexpr (is_gather_chain<Chain>()) {
        const bool streamed = (g.n_tiles & kStreamFlag) != 0u;
        if constexpr (strip_capable<Chain>()) {
            if (g.tiles_x == 0u) {                       // wave uniform: the launcher chose the strip form
                const u32 first_late = g.n_tiles & ~(kStreamFlag | kAnyPitchFlag);
                if ((g.n_tiles & kAnyPitchFlag) != 0u) {
                    if (streamed) strip_body<Chain, true, true>(p, first_late);
                    else strip_body<Chain, false, true>(p, first_late);
                } else {
                    if (streamed) strip_body<Chain, true, false>(p, first_late);
                    else strip_body<Chain, false, false>(p, first_late);
                }
                return;
            }
        }
        if constexpr (writer_streams<Chain>()) {
            if (streamed) { gather_body<Chain, FKD_GATHER_XI, FKD_GATHER_YI, true>(p, g); return; }
        }
        gather_body<Chain, FKD_GATHER_XI, FKD_GATHER_YI, false>(p, g);
    }
    else rows_auto_body<Chain, RowsConfig<Chain>::V, RowsConfig<Chain>::ROWS, rows_in_bands<Chain>(), kRowsLines>(p, 0u, &g);
}
// The module's other kernels, 1 to 6 (nothing for chains that have no such kernel).  Bilinear kernel: gather_form's forms 1 and 2, and 3 the
// strip form with its stores on line boundaries.  Rows kernel: 1 the kernel for small outputs, 2 and 3 those for planes without gaps (3: small
// outputs), 4 and 5 the chain's own and 2 for launches of few workgroups, with half the rows per thread, as 1 and 3 have, and 6 is 1 for larger ones (rows_few_blocks;
// compiled at run time, NV12 to float3 240x410 2.3 -> 2.1 us, 2000x1500 8.2 -> 7.6, RGB to P010 1804x218 2.9 -> 2.3).
template <class Chain, int WHICH> __device__ __forceinline__ void jit_other_body(const typename Chain::Params& p, const TileGeom& g) {
    if constexpr (IsDivergent<Chain>::value) {
    } else if constexpr (is_gather_chain<Chain>()) {
        if constexpr (WHICH < 3) gather_body<Chain, WHICH, 1, false>(p, g);
        else if constexpr (WHICH == 3 && strip_capable<Chain>()) {
            // (two column tables in LDS, 22.5 KB, where the kernels compiled ahead of time have one; with one for both, one image to 331x12001
            // took 13.1 us as before, to 639x4003 8.35 as before, and to 255x12001 10.4 instead of 9.9)
            if ((g.n_tiles & kStreamFlag) != 0u) strip_lines_body<Chain, true, 64>(p);
            else strip_lines_body<Chain, false, 64>(p);
        }
    } else {
        constexpr int V = RowsConfig<Chain>::V, ROWS = RowsConfig<Chain>::ROWS, HALF = ROWS > 1 ? ROWS / 2 : ROWS;
        if constexpr (WHICH == 1) rows_auto_body<Chain, V, HALF, rows_in_bands<Chain>(), kRowsSmall>(p, 0u, &g);
        else if constexpr (WHICH == 6) { if constexpr (ROWS > 1) rows_auto_body<Chain, V, ROWS, rows_in_bands<Chain>(), kRowsSmall>(p, 0u, &g); }
        else if constexpr (WHICH == 4) { if constexpr (ROWS > 1) rows_auto_body<Chain, V, HALF, rows_in_bands<Chain>(), kRowsLines>(p, 0u, &g); }
        else if constexpr (rows_have_flat<Chain>()) {
            if constexpr (WHICH != 5 || ROWS > 1) flat_body<Chain, V, WHICH == 2 ? ROWS : HALF, WHICH == 3>(p);
        }
    }
}

} // namespace fkd
