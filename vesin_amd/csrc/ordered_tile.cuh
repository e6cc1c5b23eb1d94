// The in-order search (ordered.cuh) with a workgroup per tile, from a list's second call on a system (ordered_by_tiles,
// policy.hpp):
//   COUNT and ORDER in one kernel (ordered_tile_kernel): the candidates of a tile are tested by the four waves, in single
//          precision (tile_test.cuh); those that some point of the tile has for a neighbour, about two thirds, are put in the
//          order of (original index, shift) in LDS, and their records go to memory in that order;
//   a scan over the points gives every point its first row;
//   WRITE  (ordered_write_kernel) takes the records as they come, write_tile.cuh does the rest.
// Against COUNT and SORT side by side, which order all candidates, and a WRITE that looks its candidates up by their place in
// that order (us, COUNT and SORT -> COUNT and ORDER; WRITE): 1,000,000 atoms of diamond, full P S d 590 -> 365; 930 -> 810;
// 100,000 points, 26 per cell, half P S d D 115 -> 64; 123 -> 78; 10,000 points, 29 per cell 30 -> 22; 40 -> 18.
#ifndef VESIN_HIP_ORDERED_TILE_CUH
#define VESIN_HIP_ORDERED_TILE_CUH

#include "ordered.cuh"
#include "tile_test.cuh"
#include "write_tile.cuh"

namespace vesin_hip {

constexpr uint32_t TILE_SORT_BITS = 64 * 1024;   // original indices that the bit set covers at a time
constexpr uint32_t TILE_SORT_ROUNDS = 2;         // and how often it is filled at most
constexpr uint32_t TILE_SORT_WORDS = TILE_SORT_BITS / 32;
constexpr uint32_t TILE_SORT_BUCKETS = ORDERED_CANDIDATES;
constexpr uint32_t TILE_SORT_OWN = ORDERED_CANDIDATES / TILE_BLOCK; // candidates of a thread
static_assert(TILE_SORT_WORDS == 8 * TILE_BLOCK && TILE_SORT_BUCKETS == TILE_SORT_OWN * TILE_BLOCK, "the threads share both evenly");

/// The stencil tables and the tile's points, as the tests in double precision take them.
struct TileCountTables: SearchTables {
    uint32_t tile_index[TILE_POINTS];
    double tile_x[TILE_POINTS], tile_y[TILE_POINTS], tile_z[TILE_POINTS];
};

constexpr uint32_t SELF_IMAGE = 1u << 31; // of a stencil entry: a half list keeps a point with this image of itself

struct TileOrderShared {
    TileCountTables tile;
    TileTests tests;
    // The stencil's entries that hold points: a bit per candidate, set where an entry starts, the entries before each unit of
    // 64 candidates, and per entry its first place in the cell-sorted arrays less the candidates before it, and its shift
    uint64_t entry_starts[ORDERED_UNITS];
    uint32_t entries_before[ORDERED_UNITS];
    uint32_t entry_place[MAX_ENTRIES];
    uint32_t entry_shift[MAX_ENTRIES]; // biased, | SELF_IMAGE
    // the candidates with a hit: in order of arrival, then (buckets) grouped
    uint32_t index[ORDERED_CANDIDATES];
    uint32_t biased[ORDERED_CANDIDATES];
    uint32_t column[ORDERED_CANDIDATES];
    union {
        struct {
            __attribute__((aligned(16))) uint32_t present[TILE_SORT_WORDS]; // one bit per original index of the round
            uint16_t before[TILE_SORT_WORDS / 4];                           // bits set before each group of four words
        } bits;
        uint32_t first[TILE_SORT_BUCKETS + 1]; // candidates per bucket, then the first of every bucket
    };
    uint32_t rows[TILE_POINTS];
    uint32_t tile_wrap[TILE_POINTS]; // packed_wrap of the tile's points
    uint32_t n_hits;
    uint32_t range[4]; // largest of: index, ~index, index of the lower half, ~index of the upper half
    uint32_t below_origin;
    uint32_t wave_total[TILE_WAVES];
};

/// Largest of the lanes' values, in the last lane.
__device__ __forceinline__ uint32_t wave_max_in_last_lane(uint32_t v) {
    v = max(v, dpp_or_zero<0x111, 0xf>(v));
    v = max(v, dpp_or_zero<0x112, 0xf>(v));
    v = max(v, dpp_or_zero<0x114, 0xf>(v));
    v = max(v, dpp_or_zero<0x118, 0xf>(v));
    v = max(v, dpp_or_zero<0x142, 0xa>(v));
    v = max(v, dpp_or_zero<0x143, 0xc>(v));
    return v;
}

/// The tile of a workgroup: every XCD walks one contiguous range of tiles, so that its L2 sees the same cells again and again
/// (workgroups are dealt to the XCDs round-robin). False, and tile 0, when there is none.
__device__ __forceinline__ bool tile_of_workgroup(uint32_t n_tiles, uint32_t& tile_id) {
    const uint32_t per_xcd = (n_tiles + N_XCD - 1) / N_XCD;
    const uint32_t within = blockIdx.x / N_XCD;
    tile_id = (blockIdx.x % N_XCD) * per_xcd + within;
    const bool there = within < per_xcd && tile_id < n_tiles;
    tile_id = there ? tile_id : 0u;
    return there;
}

/// The range of the original indices of candidates with a hit, and of each half of the index space.
struct TileRange {
    uint32_t highest, not_lowest, lower_highest, not_upper_lowest;
    uint32_t half;
};

/// The candidates with a hit of R units, to LDS in order of arrival.
template <int R>
__device__ __forceinline__ void keep_hits(
    TileOrderShared& sh, int lane, const uint32_t (&column)[R], const uint32_t (&index)[R], const uint32_t (&biased)[R], TileRange& range
) {
    uint64_t mask[R];
    uint32_t found = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        mask[r] = __ballot(column[r] != 0);
        found += __popcll(mask[r]);
    }
    uint32_t base = 0;
    if (lane == 0) {
        base = atomicAdd(&sh.n_hits, found);
    }
    base = uniform(base);
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (column[r] != 0) {
            const uint32_t slot = base + rank_in_mask(mask[r]);
            sh.index[slot] = index[r];
            sh.biased[slot] = biased[r];
            sh.column[slot] = column[r];
            const bool lower = index[r] < range.half;
            range.highest = max(range.highest, index[r]);
            range.not_lowest = max(range.not_lowest, ~index[r]);
            range.lower_highest = max(range.lower_highest, lower ? index[r] : 0u);
            range.not_upper_lowest = max(range.not_upper_lowest, lower ? 0u : ~index[r]);
        }
        base += __popcll(mask[r]);
    }
}

/// A wave's R units of candidates (wave, wave + TILE_WAVES, ...) against the tile's points, in single precision but for pairs
/// next to the cutoff.
template <int R, bool FULL>
__device__ __forceinline__ void count_units(
    TileOrderShared& sh, const SortedPoints& sorted, const GridParams& g, uint32_t wave, uint32_t n_candidates, uint32_t first_i,
    uint32_t n_i, int lane, bool& out_of_range, TileRange& range
) {
    TestCandidates<R> c;
    uint32_t index[R], biased[R], at[R];
    bool unshifted[R];
    const double ox = sh.tests.origin[0];
    const double oy = sh.tests.origin[1];
    const double oz = sh.tests.origin[2];
    SortedPoint point[R];
    uint32_t entry_shift[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t unit = wave + r * TILE_WAVES;
        // (lanes past the last candidate read the last one)
        const uint32_t k = min(unit * WAVE + lane, n_candidates - 1);
        const uint64_t starts = uniform(sh.entry_starts[unit]);
        const uint32_t before = uniform(sh.entries_before[unit]) + static_cast<uint32_t>(starts & 1u) - 1u;
        const uint32_t entry = before + rank_in_mask(starts >> 1);
        at[r] = sh.entry_place[entry] + k;
        entry_shift[r] = sh.entry_shift[entry];
        point[r] = sorted.p[at[r]];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const bool valid = (wave + r * TILE_WAVES) * WAVE + lane < n_candidates;
        index[r] = point[r].index;
        biased[r] = (entry_shift[r] & ~SELF_IMAGE) - point[r].wrap;
        double x = point[r].x - ox;
        double y = point[r].y - oy;
        double z = point[r].z - oz;
        if (__ballot(biased[r] != NO_SHIFT) != 0) {
            const int32_t bx = static_cast<int32_t>((biased[r] >> 20) & 0x3ffu) - 512;
            const int32_t by = static_cast<int32_t>((biased[r] >> 10) & 0x3ffu) - 512;
            const int32_t bz = static_cast<int32_t>(biased[r] & 0x3ffu) - 512;
            out_of_range = out_of_range || beyond(bx, by, bz, ORDERED_SHIFT_LIMIT);
            double tx, ty, tz;
            shift_vector(g, bx, by, bz, tx, ty, tz);
            x += tx;
            y += ty;
            z += tz;
        }
        c.x[r] = valid ? static_cast<float>(x) : NOT_THERE;
        c.y[r] = valid ? static_cast<float>(y) : NOT_THERE;
        c.z[r] = valid ? static_cast<float>(z) : NOT_THERE;
        if (!FULL) {
            // one orientation of every pair: the smaller index first; a point with its own image under the rule of the
            // reference (the total shift of such a pair is the cell shift)
            c.limit[r] = index[r] + ((entry_shift[r] & SELF_IMAGE) != 0 ? 1u : 0u);
        }
        unshifted[r] = valid && (entry_shift[r] & ~SELF_IMAGE) == NO_SHIFT;
    }
    uint32_t column[R];
    uint32_t rows;
    if (test_tile<R, FULL>(sh.tests, sh.tile.tile_index, n_i, c, column, rows) != 0) {
        resolve_tile<R, FULL>(sh.tests, sh.tile.tile_index, n_i, c, column, rows, [&](int r, uint32_t p) {
            // (the candidate is read again; every field of the sum stays inside its ten bits, operands within +-255)
            const SortedPoint candidate = sorted.p[at[r]];
            const uint32_t shift = biased[r] + sh.tile_wrap[p];
            double tx, ty, tz;
            shift_vector(
                g, static_cast<int32_t>((shift >> 20) & 0x3ffu) - 512, static_cast<int32_t>((shift >> 10) & 0x3ffu) - 512,
                static_cast<int32_t>(shift & 0x3ffu) - 512, tx, ty, tz
            );
            const double vx = (candidate.x - sh.tile.tile_x[p]) + tx;
            const double vy = (candidate.y - sh.tile.tile_y[p]) + ty;
            const double vz = (candidate.z - sh.tile.tile_z[p]) + tz;
            return vx * vx + vy * vy + vz * vz < g.cutoff2;
        });
    }
    if (FULL) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            // a point is no neighbour of itself (of its images it is)
            const uint32_t own = at[r] - first_i;
            if (unshifted[r] && own < n_i) {
                const uint32_t bit = 1u << (n_i - 1 - own);
                if ((column[r] & bit) != 0) {
                    column[r] &= ~bit;
                    atomicSub(&sh.rows[own], 1u);
                }
            }
        }
    }
    if (static_cast<uint32_t>(lane) < n_i && rows != 0) {
        atomicAdd(&sh.rows[lane], rows);
    }
    keep_hits<R>(sh, lane, column, index, biased, range);
}

/// COUNT and ORDER. Bound by its vector instructions, which are 86 % of what the compute units can issue (1,000,000 atoms of
/// diamond, 365 us): two thirds of them tests, the rest the order. Six workgroups per compute unit, 15 % slower with five. The
/// places come from a bit per original index while two rounds of 65,536 indices cover the tile, and from buckets otherwise:
/// indices without order take as long either way, runs of consecutive ones crowd a few buckets (44 % slower with one round).
template <bool FULL>
__global__ __launch_bounds__(TILE_BLOCK, 6) void ordered_tile_kernel(OrderedArgs args, GridParams g) {
    constexpr int R = ORDERED_R;
    __shared__ TileOrderShared sh;
    const int lane = lane_id();
    const uint32_t wave = uniform(threadIdx.x / WAVE);
    uint32_t tile_id;
    if (!tile_of_workgroup(static_cast<uint32_t>(args.cell_scan[g.n_cells] >> 32), tile_id)) {
        return;
    }
    const Tile tile = args.tiles[tile_id];
    const SortedPoints& sorted = args.sorted;
    const uint32_t first_i = tile.first;
    const uint32_t n_i = uniform(tile.count);
    const bool tile_wrapped = (tile.wrapped & 1u) != 0;
    const int32_t span_y = 2 * g.s[1] + 1;
    const int32_t span_z = 2 * g.s[2] + 1;
    const uint32_t n_stencil = static_cast<uint32_t>(2 * g.s[0] + 1) * span_y * span_z; // (at most MAX_ENTRIES: the host)
    bool out_of_range = false;
    if (wave == 0) {
        const int32_t cx = tile.cell % g.n[0];
        const int32_t cy = (tile.cell / g.n[0]) % g.n[1];
        const int32_t cz = tile.cell / (g.n[0] * g.n[1]);
        fill_stencil_tables(sh.tile, lane, 0, n_stencil, cx, cy, cz, span_y, span_z, g, args.cell_scan);
        if (lane < ORDERED_UNITS) {
            sh.entry_starts[lane] = 0;
        }
        wave_sync();
        // (a lane per entry: MAX_ENTRIES are as many as a wave has lanes)
        uint32_t before = 0;
        bool filled = false;
        if (static_cast<uint32_t>(lane) < n_stencil) {
            before = sh.tile.ent_prefix[lane];
            filled = sh.tile.ent_prefix[lane + 1] != before;
        }
        const uint32_t entry = rank_in_mask(__ballot(filled));
        if (filled && before < ORDERED_CANDIDATES) {
            int32_t qx, qy, qz;
            unpack_shift(sh.tile.ent_shift[lane], qx, qy, qz);
            sh.entry_place[entry] = sh.tile.ent_start[lane] - before;
            sh.entry_shift[entry] =
                biased_shift(qx, qy, qz) | ((qx | qy | qz) != 0 && half_keeps_self_image(qx, qy, qz) ? SELF_IMAGE : 0u);
            atomicOr(reinterpret_cast<uint32_t*>(sh.entry_starts) + before / 32, 1u << (before % 32));
        }
        wave_sync();
        const uint32_t starts = lane < ORDERED_UNITS ? __popcll(sh.entry_starts[lane]) : 0u;
        const uint32_t through = wave_inclusive_scan(starts);
        if (lane < ORDERED_UNITS) {
            sh.entries_before[lane] = through - starts;
        }
    } else if (wave == 1) {
        SortedPoint point = {0.0, 0.0, 0.0, 0u, 0u};
        int32_t wx = 0, wy = 0, wz = 0;
        if (static_cast<uint32_t>(lane) < n_i) {
            const uint32_t at = first_i + lane;
            point = sorted.p[at];
            wx = sorted.wx[at];
            wy = sorted.wy[at];
            wz = sorted.wz[at];
            out_of_range = beyond(wx, wy, wz, ORDERED_SHIFT_LIMIT);
            sh.tile.tile_index[lane] = point.index;
            sh.tile.tile_x[lane] = point.x;
            sh.tile.tile_y[lane] = point.y;
            sh.tile.tile_z[lane] = point.z;
            sh.tile_wrap[lane] = point.wrap;
            sh.rows[lane] = 0;
        }
        prepare_tile_tests(sh.tests, g, lane, n_i, point.x, point.y, point.z, wx, wy, wz, args.double_only);
        if (lane < 4) {
            sh.range[lane] = 0;
        }
        if (lane == 0) {
            sh.n_hits = 0;
            sh.below_origin = 0;
        }
    }
    __syncthreads();
    const uint32_t n_candidates = uniform(sh.tile.n_candidates);
    const uint32_t n_units = (n_candidates + WAVE - 1) / WAVE;
    if (threadIdx.x == 0 && n_candidates > __atomic_load_n(&args.status->max_candidates, __ATOMIC_RELAXED)) {
        atomicMax(&args.status->max_candidates, n_candidates);
    }
    if (n_candidates > ORDERED_CANDIDATES) {
        return; // the host does not use this path for such a tile: nothing to count, nothing may be written
    }

    // ---- COUNT: the waves take the units of 64 candidates in turn
    TileRange range = {0u, 0u, 0u, 0u, g.n_points / 2};
    if (uniform(sh.tests.usable) != 0) {
        const uint32_t own_units = n_units > wave ? (n_units - wave + TILE_WAVES - 1) / TILE_WAVES : 0u;
        switch (own_units) {
        case 0:
            break;
        case 1:
            count_units<1, FULL>(sh, sorted, g, wave, n_candidates, first_i, n_i, lane, out_of_range, range);
            break;
        case 2:
            count_units<2, FULL>(sh, sorted, g, wave, n_candidates, first_i, n_i, lane, out_of_range, range);
            break;
        case 3:
            count_units<3, FULL>(sh, sorted, g, wave, n_candidates, first_i, n_i, lane, out_of_range, range);
            break;
        default:
            count_units<4, FULL>(sh, sorted, g, wave, n_candidates, first_i, n_i, lane, out_of_range, range);
        }
    } else {
        if (args.report_order != 0 && threadIdx.x == 0) {
            atomicAdd(&args.status->in_double, 1u);
        }
        uint32_t rows = 0;
        for (uint32_t unit = wave; unit < n_units; unit += TILE_WAVES) {
            uint32_t column[1], at[1], original[1], biased[1];
            if (tile_wrapped) {
                ordered_sweep_pair<FULL, true, 1>(
                    sh.tile, sorted, g, unit, n_stencil, n_candidates, first_i, n_i, lane, column, rows, out_of_range, at, original, biased
                );
            } else {
                ordered_sweep_pair<FULL, false, 1>(
                    sh.tile, sorted, g, unit, n_stencil, n_candidates, first_i, n_i, lane, column, rows, out_of_range, at, original, biased
                );
            }
            keep_hits<1>(sh, lane, column, original, biased, range);
        }
        if (static_cast<uint32_t>(lane) < n_i && rows != 0) {
            atomicAdd(&sh.rows[lane], rows);
        }
    }
    if (__ballot(out_of_range) != 0 && lane == 0) {
        atomicAdd(&args.status->unsuitable, 1u);
    }
    // (systems that one round of the bit set covers need no range)
    const bool one_round = g.n_points <= TILE_SORT_BITS;
    if (!one_round) {
        range.highest = wave_max_in_last_lane(range.highest);
        range.not_lowest = wave_max_in_last_lane(range.not_lowest);
        range.lower_highest = wave_max_in_last_lane(range.lower_highest);
        range.not_upper_lowest = wave_max_in_last_lane(range.not_upper_lowest);
        if (lane == WAVE - 1) {
            atomicMax(&sh.range[0], range.highest);
            atomicMax(&sh.range[1], range.not_lowest);
            atomicMax(&sh.range[2], range.lower_highest);
            atomicMax(&sh.range[3], range.not_upper_lowest);
        }
    }
    __syncthreads();

    if (wave == 0) {
        uint32_t rows = 0;
        if (static_cast<uint32_t>(lane) < n_i) {
            rows = sh.rows[lane];
            args.rows_of_point[sh.tile.tile_index[lane]] = rows;
        }
        const uint32_t most = read_lane(wave_max_in_last_lane(rows), WAVE - 1);
        if (lane == 0 && most > __atomic_load_n(&args.status->max_rows, __ATOMIC_RELAXED)) {
            atomicMax(&args.status->max_rows, most);
        }
    }
    const uint32_t n = uniform(sh.n_hits);
    if (threadIdx.x == 0) {
        args.candidates_of_item[tile_id] = n;
    }
    if (n == 0) {
        return;
    }

    // ---- ORDER
    CandidateRecord* records = args.records + static_cast<size_t>(tile_id) * ORDERED_CANDIDATES;
    CandidateRecord own[TILE_SORT_OWN];
#pragma unroll
    for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
        const uint32_t k = u * TILE_BLOCK + threadIdx.x;
        own[u] = CandidateRecord{0u, 0u, 0u};
        if (k < n) {
            own[u] = CandidateRecord{sh.column[k], sh.index[k], sh.biased[k]};
        }
    }
    uint32_t lowest = 0;
    uint32_t highest = g.n_points - 1;
    uint32_t origin = 0;
    uint32_t last = highest; // of the window
    bool window = true;
    if (!one_round) {
        highest = uniform(sh.range[0]);
        lowest = ~uniform(sh.range[1]);
        const uint32_t upper_lowest = ~uniform(sh.range[3]);
        const uint32_t lower_highest = uniform(sh.range[2]);
        const uint32_t half = g.n_points / 2;
        constexpr uint32_t WINDOW = TILE_SORT_ROUNDS * TILE_SORT_BITS;
        origin = lowest;
        last = highest - lowest;
        if (last >= WINDOW && highest >= half && lowest < half &&
            static_cast<uint64_t>(g.n_points - upper_lowest) + lower_highest < WINDOW) {
            origin = upper_lowest;
            last = (g.n_points - upper_lowest) + lower_highest;
        }
        window = last < WINDOW;
    }
    // a point can only be seen twice when the stencil wraps around the box along some direction
    for (int d = 0; d < 3; d++) {
        window = window && !(g.periodic[d] && g.n[d] < 2 * g.s[d] + 1);
    }
    if (args.report_order != 0 && threadIdx.x == 0) {
        atomicAdd(window ? &args.status->windowed : &args.status->bucketed, 1u);
        atomicMax(&args.status->max_hits, n);
    }
    if (window) {
        uint32_t offset[TILE_SORT_OWN];
        uint32_t wrapped_around = 0;
#pragma unroll
        for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
            const uint32_t k = u * TILE_BLOCK + threadIdx.x;
            offset[u] = 0xFFFFFFFFu;
            if (k < n) {
                offset[u] = own[u].index >= origin ? own[u].index - origin : (g.n_points - origin) + own[u].index;
            }
        }
        if (origin != lowest) {
#pragma unroll
            for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
                wrapped_around += __popcll(__ballot(u * TILE_BLOCK + threadIdx.x < n && own[u].index < origin));
            }
            if (lane == 0) {
                atomicAdd(&sh.below_origin, wrapped_around);
            }
        }
        uint32_t carried = 0;
        for (uint32_t round = 0; round <= last / TILE_SORT_BITS; round++) {
            const uint32_t n_groups = (round < last / TILE_SORT_BITS ? TILE_SORT_BITS - 1 : last % TILE_SORT_BITS) / 128 + 1;
            if (round != 0) {
                __syncthreads();
            }
            for (uint32_t group = threadIdx.x; group < n_groups; group += TILE_BLOCK) {
                *reinterpret_cast<uint4*>(&sh.bits.present[4 * group]) = uint4{0u, 0u, 0u, 0u};
            }
            __syncthreads();
#pragma unroll
            for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
                if (u * TILE_BLOCK < n && offset[u] / TILE_SORT_BITS == round) {
                    const uint32_t here = offset[u] % TILE_SORT_BITS;
                    atomicOr(&sh.bits.present[here / 32], 1u << (here % 32));
                }
            }
            __syncthreads();
            // a thread has two groups of four words
            uint32_t first_group = 0, second_group = 0;
            if (2 * threadIdx.x < n_groups) {
                const uint4 a = *reinterpret_cast<const uint4*>(&sh.bits.present[8 * threadIdx.x]);
                first_group = __popc(a.x) + __popc(a.y) + __popc(a.z) + __popc(a.w);
            }
            if (2 * threadIdx.x + 1 < n_groups) {
                const uint4 b = *reinterpret_cast<const uint4*>(&sh.bits.present[8 * threadIdx.x + 4]);
                second_group = __popc(b.x) + __popc(b.y) + __popc(b.z) + __popc(b.w);
            }
            const uint32_t through = wave_inclusive_scan(first_group + second_group);
            if (lane == WAVE - 1) {
                sh.wave_total[wave] = through;
            }
            __syncthreads();
            uint32_t before = carried + through - first_group - second_group;
#pragma unroll
            for (uint32_t w = 0; w < TILE_WAVES; w++) {
                const uint32_t total = sh.wave_total[w];
                before += w < wave ? total : 0u;
                carried += total;
            }
            // (two 16-bit numbers in one store)
            reinterpret_cast<uint32_t*>(sh.bits.before)[threadIdx.x] = before | ((before + first_group) << 16);
            __syncthreads();
            const uint32_t below = origin != lowest ? uniform(sh.below_origin) : 0u;
            const uint32_t in_window_first = n - below;
#pragma unroll
            for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
                if (u * TILE_BLOCK < n && offset[u] / TILE_SORT_BITS == round) {
                    const uint32_t here = offset[u] % TILE_SORT_BITS;
                    const uint32_t word = here / 32;
                    const uint4 words = *reinterpret_cast<const uint4*>(&sh.bits.present[word & ~3u]);
                    uint32_t place = sh.bits.before[word / 4];
                    place += (word % 4 > 0) ? __popc(words.x) : 0;
                    place += (word % 4 > 1) ? __popc(words.y) : 0;
                    place += (word % 4 > 2) ? __popc(words.z) : 0;
                    const uint32_t mine = word % 4 == 0 ? words.x : word % 4 == 1 ? words.y : word % 4 == 2 ? words.z : words.w;
                    place += __popc(mine & ((1u << (here % 32)) - 1u));
                    // the window's order starts at the origin, the order of the indices with those that wrapped around
                    place = place >= in_window_first ? place - in_window_first : place + below;
                    records[min(place, ORDERED_CANDIDATES - 1)] = own[u];
                }
            }
        }
        return;
    }

    const float per_index = static_cast<float>(TILE_SORT_BUCKETS) / (static_cast<float>(highest - lowest) + 1.0f);
    auto bucket_of = [&](uint32_t i) {
        return min(TILE_SORT_BUCKETS - 1, static_cast<uint32_t>(static_cast<float>(i - lowest) * per_index));
    };
    for (uint32_t b = threadIdx.x; b <= TILE_SORT_BUCKETS; b += TILE_BLOCK) {
        sh.first[b] = 0;
    }
    __syncthreads();
    uint32_t bucket[TILE_SORT_OWN], arrival[TILE_SORT_OWN];
#pragma unroll
    for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
        bucket[u] = bucket_of(own[u].index);
        arrival[u] = u * TILE_BLOCK + threadIdx.x < n ? atomicAdd(&sh.first[bucket[u]], 1u) : 0u;
    }
    __syncthreads();
    uint32_t in_bucket[TILE_SORT_OWN];
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t b = 0; b < TILE_SORT_OWN; b++) {
        in_bucket[b] = sh.first[TILE_SORT_OWN * threadIdx.x + b];
        mine += in_bucket[b];
    }
    const uint32_t through = wave_inclusive_scan(mine);
    if (lane == WAVE - 1) {
        sh.wave_total[wave] = through;
    }
    __syncthreads();
    uint32_t before = through - mine;
    for (uint32_t w = 0; w < wave; w++) {
        before += sh.wave_total[w];
    }
#pragma unroll
    for (uint32_t b = 0; b < TILE_SORT_OWN; b++) {
        sh.first[TILE_SORT_OWN * threadIdx.x + b] = before;
        before += in_bucket[b];
    }
    if (threadIdx.x == TILE_BLOCK - 1) {
        sh.first[TILE_SORT_BUCKETS] = before; // = n
    }
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
        if (u * TILE_BLOCK + threadIdx.x < n) {
            const uint32_t slot = sh.first[bucket[u]] + arrival[u];
            sh.index[slot] = own[u].index;
            sh.biased[slot] = own[u].biased;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < TILE_SORT_OWN; u++) {
        if (u * TILE_BLOCK + threadIdx.x < n) {
            uint32_t place = sh.first[bucket[u]];
            const uint32_t end = sh.first[bucket[u] + 1];
            for (uint32_t other = place; other < end; other++) {
                const uint32_t theirs = sh.index[other];
                // (the images of one point differ in their shifts)
                place += theirs < own[u].index || (theirs == own[u].index && sh.biased[other] < own[u].biased) ? 1u : 0u;
            }
            records[place] = own[u];
        }
    }
}

/// WRITE. Bound by its stores: 1,000,000 atoms of diamond, P S d, 810 us, 460 without them; see tile_stores, policy.hpp.
template <bool STAGED, TileStores STORES>
__global__ __launch_bounds__(TILE_BLOCK, STAGED ? 4 : 5) void ordered_write_kernel(OrderedArgs args, GridParams g) {
    __shared__ TileWriteShared<STAGED> sh;
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    const uint32_t wave = uniform(threadIdx.x / WAVE);
    // What the first chunk needs comes through a chain of loads (record, point), each of which takes microseconds beside
    // the stores of the other workgroups: all that does not depend on another load is asked for at once (there is room for
    // ORDERED_CANDIDATES records per tile, whatever the tile uses).
    const uint32_t n_tiles = static_cast<uint32_t>(args.cell_scan[g.n_cells] >> 32);
    uint32_t tile_id;
    const bool there = tile_of_workgroup(n_tiles, tile_id);
    const CandidateRecord* records = args.records + static_cast<size_t>(tile_id) * ORDERED_CANDIDATES;
    constexpr uint32_t OWN = (TILE_CHUNK + TILE_BLOCK - 1) / TILE_BLOCK; // candidates of a chunk that a thread brings
    CandidateRecord record[OWN];
    double x[OWN], y[OWN], z[OWN];
    auto load_records = [&](uint32_t first) {
#pragma unroll
        for (uint32_t u = 0; u < OWN; u++) {
            record[u] = records[min(first + u * TILE_BLOCK + threadIdx.x, ORDERED_CANDIDATES - 1)];
        }
    };
    load_records(0);
    const uint32_t max_rows = args.status->max_rows;
    const uint32_t max_candidates = args.status->max_candidates;
    const uint32_t unsuitable = args.status->unsuitable;
    const uint64_t total_rows = args.first_row[g.n_points];
    const uint32_t n_or_garbage = args.candidates_of_item[tile_id];
    const Tile tile = args.tiles[tile_id];
    if (args.publish_to != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
        OrderedHostStatus report;
        report.found = *args.status;
        report.total_rows = total_rows;
        report.first_bad_coordinate = args.build_status->first_bad_coordinate;
        report.n_tiles = n_tiles;
        *args.publish_to = report;
    }
    const bool suitable =
        max_rows <= ORDERED_MAX_ROWS && max_candidates <= ORDERED_CANDIDATES && unsuitable == 0 && total_rows <= args.capacity;
    if (!there || (args.guarded != 0 && !suitable)) {
        return;
    }
    const uint32_t n = uniform(n_or_garbage);
    const uint32_t n_i = uniform(tile.count);
    auto load_points = [&](uint32_t first) {
#pragma unroll
        for (uint32_t u = 0; u < OWN; u++) {
            const uint32_t k = u * TILE_BLOCK + threadIdx.x;
            if (k >= TILE_CHUNK || first + k >= n) {
                record[u] = CandidateRecord{0u, 0u, NO_SHIFT};
            }
            const double* point = args.points + 3 * static_cast<size_t>(record[u].index);
            x[u] = point[0];
            y[u] = point[1];
            z[u] = point[2];
        }
    };
    load_points(0);
    const bool moved = load_tile(sh, args.sorted, tile.first, n_i, args.first_row);
    for (uint32_t first = 0; first < n; first += TILE_CHUNK) {
        if (first != 0) {
            load_records(first);
            load_points(first);
            __syncthreads();
        }
        bool shifted = moved;
#pragma unroll
        for (uint32_t u = 0; u < OWN; u++) {
            const uint32_t k = u * TILE_BLOCK + threadIdx.x;
            if (k < TILE_CHUNK) {
                sh.x[k] = x[u];
                sh.y[k] = y[u];
                sh.z[k] = z[u];
                sh.index[k] = record[u].index;
                sh.biased[k] = record[u].biased;
                sh.column[k] = record[u].column;
            }
            shifted = shifted || record[u].biased != NO_SHIFT;
        }
        const uint32_t units_here = (min(n - first, TILE_CHUNK) + WAVE - 1) / WAVE;
        if (__syncthreads_or(shifted) != 0) {
            write_tile_chunk<true, STAGED, STORES>(sh, wave, g, args.out, n_i, units_here, n > TILE_CHUNK, lane);
        } else {
            write_tile_chunk<false, STAGED, STORES>(sh, wave, g, args.out, n_i, units_here, n > TILE_CHUNK, lane);
        }
    }
}

} // namespace vesin_hip

#endif
