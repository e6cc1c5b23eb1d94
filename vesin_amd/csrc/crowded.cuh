// In-order search of systems that ordered.cuh does not cover because their cells are crowded (more than 1024 candidates
// around a tile, or more than 256 rows of a point: dense clusters, cutoffs of several interatomic distances) or because
// there are too many cells for its records of a fixed size (clusters in a wide, mostly empty box).
//
// The scheme is the same: every tile tests its points against the whole stencil, so every row is found by the tile of
// its first point; candidates in the order of (original index, shift) make the hits of a point, taken in that order,
// its rows in final order. What differs is how the work is laid out, so that nothing is of a fixed size:
//   MEASURE  every cell that holds points counts its candidates and takes room for them, and for one word per
//            candidate and tile, from a running total (where the room lies in memory does not enter the result);
//   SORT     one workgroup per cell, not per tile: the tiles of a cell share their candidates. Candidates are grouped in
//            LDS by ranges of the original index (buckets), then ranked inside their bucket, and go to memory as
//            (position in the cell-sorted arrays, biased shift less the wrap of the first point) in final order;
//   COUNT    one workgroup per tile, the candidates dealt to its four waves: hit columns in the order of the candidates,
//            rows of every point;
//   a scan over the points gives every point its first row;
//   WRITE    one workgroup per tile: write_tile.cuh.
// A point may have any number of rows; a cell at most CROWDED_LARGE candidates (their sort takes the LDS of a compute
// unit then). Beyond that, and for shifts or wraps beyond +-255, the host falls back to the radix sort.
//
// Measured per call, full lists, radix sort -> this: 500,000 points in 50 clusters (82 M rows, P d) 13.2 -> 1.44 ms, (P S d D)
// 18.5 -> 2.35 ms; 195,112 atoms of diamond, cutoff 6.5 (1480 candidates per tile, P S d) 6.10 -> 1.06 ms; 13,824 atoms, cutoff
// 5.5, 378 -> 171 us; liquids of 0.1 points per unit of volume, cutoff 7: 20,000 points 560 -> 182 us, 2,000 points 216 -> 152
// us. On systems that
// ordered_tile.cuh covers it is the slower one: it orders all candidates of a cell, where that one orders those with a hit
// (1,000,000 atoms of diamond 1.26 against 1.93 ms, 100,000 points, half P S d D, 210 against 245 us).
//
// Arithmetic and order as in ordered.cuh (vesin/src/cpu_cell_list.cpp:135-138, vesin/src/types.hpp:232-243).
#ifndef VESIN_HIP_CROWDED_CUH
#define VESIN_HIP_CROWDED_CUH

#include "ordered.cuh"
#include "tile_test.cuh"
#include "write_tile.cuh"

namespace vesin_hip {

constexpr int CROWDED_WAVES = 4;
constexpr int CROWDED_BLOCK = CROWDED_WAVES * WAVE;
constexpr uint32_t CROWDED_SMALL = 2048;   // candidates that the usual sorting kernel takes (29 KB of LDS)
constexpr uint32_t CROWDED_LARGE = 8192;   // and the one for the most crowded cells (115 KB)
constexpr int CROWDED_SORT_BLOCK = 512;    // threads of the latter
constexpr uint32_t CROWDED_BUCKET = 64;    // keys of a bucket that is left as it is
constexpr uint32_t CROWDED_LEVELS = 6;     // times that the buckets are shared out again at most
static_assert(CROWDED_BUCKET >= MAX_ENTRIES, "the images of one point share a bucket, whatever it is shared out into");

/// A candidate, in the order of (original index, shift).
struct CrowdedCandidate {
    uint32_t at;     // position in the cell-sorted arrays
    uint32_t biased; // cell shift less the wrap of the candidate, biased (see biased_shift)
};

/// What a cell was given, at the number of its first tile.
struct CrowdedCell {
    uint32_t candidates;      // 0: no room (see CrowdedStatus::overflow), or too many
    uint32_t first_candidate; // in units of 64
    uint32_t first_column;    // in units of 64, of the cell's first tile; the next tiles follow
    uint32_t padding;
};

/// Device memory, cleared before MEASURE.
struct CrowdedStatus {
    unsigned long long used; // units of 64 candidates taken | units of 64 hit columns taken << 32
    unsigned int max_candidates;
    unsigned int unsuitable; // a shift or wrap outside of the key's range
    unsigned int overflow;   // cells that found no room left
    unsigned int in_double;  // tiles whose pairs were all tested in double precision (where it is reported)
};

/// What the host reads after COUNT and the scan (pinned host memory).
struct CrowdedHostStatus {
    CrowdedStatus found;
    unsigned long long total_rows;
    unsigned int first_bad_coordinate;
    unsigned int n_tiles;
};

struct CrowdedArgs {
    SortedPoints sorted;
    const uint64_t* cell_scan;
    const Tile* tiles;
    CrowdedCell* cells;           // [tile slots]
    CrowdedCandidate* candidates; // [candidate_units * 64]
    uint32_t* columns;            // [column_units * 64]
    uint32_t candidate_units;
    uint32_t column_units;
    CrowdedStatus* status;
    uint32_t* rows_of_point;      // COUNT: [n_points], by original index
    const uint64_t* first_row;    // WRITE: [n_points + 1], their exclusive scan
    uint64_t capacity;            // WRITE: rows that the output arrays hold; nothing is written when there are more
    SearchOutputs out;
    uint32_t double_only;         // COUNT: not zero: every pair is tested in double precision (for tests)
    uint32_t report;              // COUNT: count the tiles where they are (an atomic on one word: for tests)
};

/// Number `turn` of the tiles that a workgroup takes (n_tiles or beyond: none): every XCD walks a contiguous range of
/// tiles, so that its L2 sees the same cells again and again (workgroups are dealt to the XCDs round-robin).
__device__ __forceinline__ uint32_t crowded_tile(uint32_t turn, uint32_t n_tiles) {
    const uint32_t per_xcd = (n_tiles + N_XCD - 1) / N_XCD;
    const uint32_t within = blockIdx.x / N_XCD + turn * (gridDim.x / N_XCD);
    const uint32_t tile = (blockIdx.x % N_XCD) * per_xcd + within;
    return within < per_xcd && tile < n_tiles ? tile : 0xFFFFFFFFu;
}

__device__ __forceinline__ uint32_t crowded_first_tile(const CrowdedArgs& args, const Tile& tile) {
    return static_cast<uint32_t>(args.cell_scan[tile.cell] >> 32);
}

__device__ __forceinline__ uint32_t fill_crowded_tables(
    SearchTables& sh, int lane, uint32_t cell, const GridParams& g, const uint64_t* __restrict__ cell_scan
) {
    const int32_t span_y = 2 * g.s[1] + 1;
    const int32_t span_z = 2 * g.s[2] + 1;
    const uint32_t n_stencil = static_cast<uint32_t>(2 * g.s[0] + 1) * span_y * span_z; // (at most MAX_ENTRIES: the host)
    fill_stencil_tables(
        sh, lane, 0, n_stencil, static_cast<int32_t>(cell % g.n[0]), static_cast<int32_t>((cell / g.n[0]) % g.n[1]),
        static_cast<int32_t>(cell / (g.n[0] * g.n[1])), span_y, span_z, g, cell_scan
    );
    return n_stencil;
}

// ---------------------------------------------------------------------------------------------------------------
// MEASURE: one thread per tile, of which the first of every cell counts. The threads of a workgroup take room together:
// one atomic each on the running total, which all compute dies share, took 1.5 ms for 44,000 cells.

__global__ __launch_bounds__(CROWDED_BLOCK) void crowded_measure_kernel(CrowdedArgs args, GridParams g) {
    __shared__ unsigned long long wave_total[CROWDED_WAVES];
    __shared__ unsigned long long taken;
    const int lane = lane_id();
    const uint32_t wave = uniform(threadIdx.x / WAVE);
    const uint32_t n_tiles = static_cast<uint32_t>(args.cell_scan[g.n_cells] >> 32);
    for (uint32_t t0 = blockIdx.x * CROWDED_BLOCK; t0 < n_tiles; t0 += gridDim.x * CROWDED_BLOCK) {
        const uint32_t t = t0 + threadIdx.x;
        uint32_t n = 0;
        uint32_t tiles_here = 0;
        if (t < n_tiles) {
            const uint32_t cell = args.tiles[t].cell;
            if (static_cast<uint32_t>(args.cell_scan[cell] >> 32) == t) {
                tiles_here = static_cast<uint32_t>(args.cell_scan[cell + 1] >> 32) - t;
                const int32_t cx = static_cast<int32_t>(cell % g.n[0]);
                const int32_t cy = static_cast<int32_t>((cell / g.n[0]) % g.n[1]);
                const int32_t cz = static_cast<int32_t>(cell / (g.n[0] * g.n[1]));
                for (int32_t dx = -g.s[0]; dx <= g.s[0]; dx++) {
                    for (int32_t dy = -g.s[1]; dy <= g.s[1]; dy++) {
                        for (int32_t dz = -g.s[2]; dz <= g.s[2]; dz++) {
                            uint32_t neighbour;
                            int32_t q[3];
                            if (stencil_neighbour(g, cx, cy, cz, dx, dy, dz, neighbour, q)) {
                                n += static_cast<uint32_t>(args.cell_scan[neighbour + 1]) -
                                     static_cast<uint32_t>(args.cell_scan[neighbour]);
                            }
                        }
                    }
                }
            }
        }
        const uint32_t n_units = n > CROWDED_LARGE ? 0u : (n + WAVE - 1) / WAVE;
        const unsigned long long wanted =
            static_cast<unsigned long long>(n_units) | (static_cast<unsigned long long>(n_units) * tiles_here << 32);
        const unsigned long long through = wave_inclusive_scan(static_cast<uint64_t>(wanted));
        __syncthreads(); // (the round before has read the totals)
        if (lane == WAVE - 1) {
            wave_total[wave] = through;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long all = 0;
            for (int w = 0; w < CROWDED_WAVES; w++) {
                all += wave_total[w];
            }
            taken = all != 0 ? atomicAdd(&args.status->used, all) : 0;
        }
        __syncthreads();
        unsigned long long mine = taken + through - wanted;
        for (uint32_t w = 0; w < wave; w++) {
            mine += wave_total[w];
        }
        if (tiles_here != 0) {
            CrowdedCell cell = {n, static_cast<uint32_t>(mine), static_cast<uint32_t>(mine >> 32), 0u};
            if (n > CROWDED_LARGE) {
                cell.candidates = 0;
            } else if (static_cast<uint64_t>(cell.first_candidate) + n_units > args.candidate_units ||
                       static_cast<uint64_t>(cell.first_column) + static_cast<uint64_t>(n_units) * tiles_here > args.column_units) {
                cell.candidates = 0;
                args.status->overflow = 1u;
            }
            args.cells[t] = cell;
        }
        uint32_t most = n;
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), offset, WAVE)));
        }
        if (lane == 0 && most > __atomic_load_n(&args.status->max_candidates, __ATOMIC_RELAXED)) {
            atomicMax(&args.status->max_candidates, most);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// SORT: bound by LDS latency and atomics. Buckets of about two candidates' indices, so that a key meets few others, where
// the indices are spread evenly; where they clump (a blob numbered in one go and some points of another, a solute numbered
// before its solvent) nearly all would share a few buckets and be compared one by one, and the range of every bucket is
// shared out again until none holds more than 64. The kernel for most cells and the one for the most crowded are apart
// because the latter's LDS leaves room for one workgroup per compute unit (clusters of 500,000 points without and with sharing
// out again: in no order 208 + 120 and 209 + 121 us, blobs numbered one after the other, each along x, 0.2 % of the points
// before them all 643 + 153 and 337 + 153 us; per call of 2,000,000 points 5.65 and 5.66 ms, 9.41 and 6.06 ms).

template <uint32_t CAPACITY, int THREADS>
struct CrowdedSortShared {
    static constexpr uint32_t BUCKETS = CAPACITY / 2;
    SearchTables tables;
    uint32_t index[CAPACITY];  // grouped by bucket
    uint32_t at[CAPACITY];
    uint32_t biased[CAPACITY];
    uint32_t first[BUCKETS + 1]; // candidates per bucket, then the first of every bucket
    uint32_t lowest, highest;
    uint32_t wide_bucket; // some bucket holds more than CROWDED_BUCKET
    uint32_t wave_total[THREADS / WAVE];
};

/// Cells of more than `MORE_THAN` and at most `CAPACITY` candidates.
template <uint32_t MORE_THAN, uint32_t CAPACITY, int THREADS>
__global__ __launch_bounds__(THREADS) void crowded_sort_kernel(CrowdedArgs args, GridParams g) {
    using Shared = CrowdedSortShared<CAPACITY, THREADS>;
    constexpr uint32_t OWN = CAPACITY / THREADS; // candidates of a thread
    constexpr uint32_t BUCKETS = Shared::BUCKETS;
    constexpr uint32_t OWN_BUCKETS = BUCKETS / THREADS;
    static_assert(OWN * THREADS == CAPACITY && OWN_BUCKETS * THREADS == BUCKETS, "the threads share everything evenly");
    __shared__ Shared sh;
    const int lane = lane_id();
    const uint32_t wave = uniform(threadIdx.x / WAVE);
    const uint32_t n_tiles = static_cast<uint32_t>(args.cell_scan[g.n_cells] >> 32);
    if (CAPACITY == CROWDED_LARGE && args.status->max_candidates <= MORE_THAN) {
        return;
    }
    for (uint32_t turn = 0;; turn++) {
        if (turn * (gridDim.x / N_XCD) + blockIdx.x / N_XCD >= (n_tiles + N_XCD - 1) / N_XCD) {
            return;
        }
        const uint32_t t = crowded_tile(turn, n_tiles);
        if (t == 0xFFFFFFFFu) {
            continue;
        }
        const Tile tile = args.tiles[t];
        if (crowded_first_tile(args, tile) != t) {
            continue;
        }
        const CrowdedCell cell = args.cells[t];
        const uint32_t n = uniform(cell.candidates);
        if (n == 0 || n <= MORE_THAN || n > CAPACITY) {
            continue;
        }
        __syncthreads(); // (the cell before is done with the LDS)
        const uint32_t n_stencil = static_cast<uint32_t>(2 * g.s[0] + 1) * (2 * g.s[1] + 1) * (2 * g.s[2] + 1);
        if (wave == 0) {
            (void)fill_crowded_tables(sh.tables, lane, tile.cell, g, args.cell_scan);
        }
        if (threadIdx.x == 0) {
            sh.lowest = 0xFFFFFFFFu;
            sh.highest = 0;
            sh.wide_bucket = 0;
        }
        for (uint32_t b = threadIdx.x; b <= BUCKETS; b += THREADS) {
            sh.first[b] = 0;
        }
        __syncthreads();

        uint32_t index[OWN], at[OWN], biased[OWN];
        uint32_t lowest = 0xFFFFFFFFu;
        uint32_t highest = 0;
        bool out_of_range = false;
#pragma unroll
        for (uint32_t u = 0; u < OWN; u++) {
            // (the kernel for the most crowded cells is better off without a branch per lane: 127 -> 121 us)
            const uint32_t own = u * THREADS + threadIdx.x;
            const uint32_t k = CAPACITY == CROWDED_LARGE ? min(own, n - 1) : own;
            index[u] = at[u] = biased[u] = 0;
            if (CAPACITY == CROWDED_LARGE ? u * THREADS < n : own < n) {
                int32_t packed;
                locate_candidate(sh.tables, n_stencil, k, at[u], packed);
                int32_t qx, qy, qz;
                unpack_shift(packed, qx, qy, qz);
                index[u] = args.sorted.p[at[u]].index;
                qx -= args.sorted.wx[at[u]];
                qy -= args.sorted.wy[at[u]];
                qz -= args.sorted.wz[at[u]];
                biased[u] = biased_shift(qx, qy, qz);
                out_of_range = out_of_range || beyond(qx, qy, qz, ORDERED_SHIFT_LIMIT);
                lowest = min(lowest, index[u]);
                highest = max(highest, index[u]);
            }
        }
        if (__ballot(out_of_range) != 0 && lane == 0) {
            atomicOr(&args.status->unsuitable, 1u);
        }
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            lowest = min(lowest, static_cast<uint32_t>(__shfl_xor(static_cast<int>(lowest), offset, WAVE)));
            highest = max(highest, static_cast<uint32_t>(__shfl_xor(static_cast<int>(highest), offset, WAVE)));
        }
        if (lane == 0) {
            atomicMin(&sh.lowest, lowest);
            atomicMax(&sh.highest, highest);
        }
        __syncthreads();
        lowest = uniform(sh.lowest);
        highest = uniform(sh.highest);
        // monotonic in the index: products of exact and rounded numbers with one factor, rounded again
        const float per_index = static_cast<float>(BUCKETS) / (static_cast<float>(highest - lowest) + 1.0f);
        auto bucket_of = [&](uint32_t i) {
            return min(BUCKETS - 1, static_cast<uint32_t>(static_cast<float>(i - lowest) * per_index));
        };
        uint32_t bucket[OWN], arrival[OWN];
#pragma unroll
        for (uint32_t u = 0; u < OWN; u++) {
            bucket[u] = bucket_of(index[u]);
        }
        uint32_t level = 0;
        for (;; level++) {
#pragma unroll
            for (uint32_t u = 0; u < OWN; u++) {
                const uint32_t k = u * THREADS + threadIdx.x;
                arrival[u] = k < n ? atomicAdd(&sh.first[bucket[u]], 1u) : 0u;
            }
            __syncthreads();
            uint32_t in_bucket[OWN_BUCKETS];
            uint32_t mine = 0;
            uint32_t most = 0;
#pragma unroll
            for (uint32_t b = 0; b < OWN_BUCKETS; b++) {
                in_bucket[b] = sh.first[OWN_BUCKETS * threadIdx.x + b];
                mine += in_bucket[b];
                most = max(most, in_bucket[b]);
            }
            const uint32_t through = wave_inclusive_scan(mine);
            if (lane == WAVE - 1) {
                sh.wave_total[wave] = through;
            }
            if (most > CROWDED_BUCKET) {
                sh.wide_bucket = 1;
            }
            __syncthreads();
            const bool share_again = uniform(sh.wide_bucket) != 0 && level < CROWDED_LEVELS;
            uint32_t before = through - mine;
            for (uint32_t w = 0; w < wave; w++) {
                before += sh.wave_total[w];
            }
#pragma unroll
            for (uint32_t b = 0; b < OWN_BUCKETS; b++) {
                sh.first[OWN_BUCKETS * threadIdx.x + b] = before;
                before += in_bucket[b];
            }
            if (threadIdx.x == THREADS - 1) {
                sh.first[BUCKETS] = before; // = n
            }
            if (!share_again) {
                break;
            }
            // Some bucket holds many: every bucket's own range of indices is shared out again among as many places as it
            // has keys, which gives an estimate of every key's rank, and the ranks two by two are the new buckets.
            // (in rolled loops on LDS that is not in use yet: 337 us in the clumped case, 346 from the registers)
            uint32_t* const low = sh.at;
            uint32_t* const high = sh.at + BUCKETS;
            for (uint32_t b = threadIdx.x; b < BUCKETS; b += THREADS) {
                low[b] = 0xFFFFFFFFu;
                high[b] = 0;
            }
#pragma unroll
            for (uint32_t u = 0; u < OWN; u++) {
                sh.index[u * THREADS + threadIdx.x] = index[u];
                sh.biased[u * THREADS + threadIdx.x] = bucket[u];
            }
            __syncthreads();
#pragma unroll 1
            for (uint32_t k = threadIdx.x; k < n; k += THREADS) { // (each thread its own candidates)
                atomicMin(&low[sh.biased[k]], sh.index[k]);
                atomicMax(&high[sh.biased[k]], sh.index[k]);
            }
            __syncthreads();
#pragma unroll 1
            for (uint32_t k = threadIdx.x; k < n; k += THREADS) {
                const uint32_t own = sh.biased[k];
                const uint32_t first = sh.first[own];
                const uint32_t keys = sh.first[own + 1] - first;
                const float per_place = static_cast<float>(keys) / (static_cast<float>(high[own] - low[own]) + 1.0f);
                const uint32_t place = static_cast<uint32_t>(static_cast<float>(sh.index[k] - low[own]) * per_place);
                sh.biased[k] = (first + min(keys - 1, place)) / 2;
            }
#pragma unroll
            for (uint32_t u = 0; u < OWN; u++) {
                bucket[u] = sh.biased[u * THREADS + threadIdx.x];
            }
            __syncthreads();
            for (uint32_t b = threadIdx.x; b <= BUCKETS; b += THREADS) {
                sh.first[b] = 0;
            }
            if (threadIdx.x == 0) {
                sh.wide_bucket = 0;
            }
            __syncthreads();
        }
        __syncthreads();
#pragma unroll
        for (uint32_t u = 0; u < OWN; u++) {
            if (u * THREADS + threadIdx.x < n) {
                const uint32_t slot = sh.first[bucket[u]] + arrival[u];
                sh.index[slot] = index[u];
                sh.at[slot] = at[u];
                sh.biased[slot] = biased[u];
            }
        }
        __syncthreads();
        CrowdedCandidate* target = args.candidates + static_cast<size_t>(cell.first_candidate) * WAVE;
        for (uint32_t slot = threadIdx.x; slot < n; slot += THREADS) {
            const uint32_t own = sh.index[slot];
            const uint32_t own_biased = sh.biased[slot];
            uint32_t own_bucket = 0;
            if (level == 0) {
                own_bucket = bucket_of(own);
            } else {
                // the last bucket that starts at the slot or before it
#pragma unroll
                for (uint32_t step = BUCKETS / 2; step > 0; step /= 2) {
                    own_bucket += sh.first[own_bucket + step] <= slot ? step : 0u;
                }
            }
            const uint32_t end = sh.first[own_bucket + 1];
            uint32_t place = sh.first[own_bucket];
            for (uint32_t other = place; other < end; other++) {
                const uint32_t theirs = sh.index[other];
                // (the images of one point differ in their shifts)
                place += theirs < own || (theirs == own && sh.biased[other] < own_biased) ? 1u : 0u;
            }
            target[place] = CrowdedCandidate{sh.at[slot], own_biased};
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// COUNT: in single precision (tile_test.cuh). Vector instructions fill two thirds of it, the rest is the latency of its
// loads and the most crowded tiles, whose candidates are dealt to four waves (they would otherwise run long after all others
// are done). In double precision -> this: clusters of 500,000 points 270 -> 250 us, 195,112 atoms at cutoff 6.5 298 -> 105 us,
// 13,824 atoms at cutoff 5.5 33 -> 17 us. Four units at a time 275 us, three 264 (registers).

struct CrowdedCountShared {
    uint32_t tile_index[TILE_POINTS];
    double tile_x[TILE_POINTS], tile_y[TILE_POINTS], tile_z[TILE_POINTS];
    int32_t tile_wx[TILE_POINTS], tile_wy[TILE_POINTS], tile_wz[TILE_POINTS];
    uint32_t rows[TILE_POINTS];
    TileTests tests;
};

/// R units of candidates (unit0, unit0 + CROWDED_WAVES, ...) against the tile's points, in single precision but for pairs next to the
/// cutoff; lane p of `own_rows` adds up the hits of point p.
template <int R, bool FULL>
__device__ __forceinline__ void crowded_count_units(
    CrowdedCountShared& sh, const SortedPoints& sorted, const GridParams& g, const CrowdedCandidate* __restrict__ candidates,
    uint32_t* __restrict__ columns, uint32_t unit0, uint32_t n, uint32_t first_i, uint32_t n_i, int lane, uint32_t& own_rows
) {
    TestCandidates<R> c;
    CrowdedCandidate candidate[R];
    SortedPoint point[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        // (lanes past the last candidate read the last one)
        candidate[r] = candidates[min((unit0 + r * CROWDED_WAVES) * WAVE + lane, n - 1)];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        point[r] = sorted.p[candidate[r].at];
    }
    auto shift_of = [&](uint32_t biased, double& tx, double& ty, double& tz) {
        shift_vector(
            g, static_cast<int32_t>((biased >> 20) & 0x3ffu) - 512, static_cast<int32_t>((biased >> 10) & 0x3ffu) - 512,
            static_cast<int32_t>(biased & 0x3ffu) - 512, tx, ty, tz
        );
    };
#pragma unroll
    for (int r = 0; r < R; r++) {
        const bool valid = (unit0 + r * CROWDED_WAVES) * WAVE + lane < n;
        double x = point[r].x - sh.tests.origin[0];
        double y = point[r].y - sh.tests.origin[1];
        double z = point[r].z - sh.tests.origin[2];
        if (__ballot(candidate[r].biased != NO_SHIFT) != 0) {
            double tx, ty, tz;
            shift_of(candidate[r].biased, tx, ty, tz);
            x += tx;
            y += ty;
            z += tz;
        }
        c.x[r] = valid ? static_cast<float>(x) : NOT_THERE;
        c.y[r] = valid ? static_cast<float>(y) : NOT_THERE;
        c.z[r] = valid ? static_cast<float>(z) : NOT_THERE;
        if (!FULL) {
            // one orientation of every pair: the smaller index first; a point with its own image under the rule of the
            // reference: the total shift of such a pair is the cell shift
            const uint32_t cell_shift = candidate[r].biased + point[r].wrap;
            const bool own_image = cell_shift != NO_SHIFT && half_keeps_self_image(
                                                                 static_cast<int32_t>((cell_shift >> 20) & 0x3ffu) - 512,
                                                                 static_cast<int32_t>((cell_shift >> 10) & 0x3ffu) - 512,
                                                                 static_cast<int32_t>(cell_shift & 0x3ffu) - 512
                                                             );
            c.limit[r] = point[r].index + (own_image ? 1u : 0u);
        }
    }
    uint32_t column[R];
    uint32_t rows;
    if (test_tile<R, FULL>(sh.tests, sh.tile_index, n_i, c, column, rows) != 0) {
        resolve_tile<R, FULL>(sh.tests, sh.tile_index, n_i, c, column, rows, [&](int r, uint32_t p) {
            const CrowdedCandidate again = candidates[min((unit0 + r * CROWDED_WAVES) * WAVE + lane, n - 1)];
            const SortedPoint there = sorted.p[again.at];
            double tx, ty, tz;
            shift_of(again.biased + packed_wrap(sh.tile_wx[p], sh.tile_wy[p], sh.tile_wz[p]), tx, ty, tz);
            const double vx = (there.x - sh.tile_x[p]) + tx;
            const double vy = (there.y - sh.tile_y[p]) + ty;
            const double vz = (there.z - sh.tile_z[p]) + tz;
            return vx * vx + vy * vy + vz * vz < g.cutoff2;
        });
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t k = (unit0 + r * CROWDED_WAVES) * WAVE + lane;
        if (FULL) {
            // a point is no neighbour of itself (of its images it is)
            const uint32_t own = candidate[r].at - first_i;
            const uint32_t bit = 1u << ((n_i - 1 - own) % 32u);
            const bool itself = k < n && own < n_i && candidate[r].biased + point[r].wrap == NO_SHIFT && (column[r] & bit) != 0;
            column[r] &= itself ? ~bit : ~0u;
            if (__ballot(itself) != 0) {
                if (itself) {
                    atomicSub(&sh.rows[own], 1u);
                }
            }
        }
        columns[k] = column[r];
    }
    own_rows += rows;
}

template <bool FULL>
__global__ __launch_bounds__(CROWDED_BLOCK, 5) void crowded_count_kernel(CrowdedArgs args, GridParams g) {
    constexpr int R = ORDERED_R;
    __shared__ CrowdedCountShared sh;
    const int lane = lane_id();
    const uint32_t wave = uniform(threadIdx.x / WAVE);
    const uint32_t n_tiles = static_cast<uint32_t>(args.cell_scan[g.n_cells] >> 32);
    for (uint32_t turn = 0;; turn++) {
        if (turn * (gridDim.x / N_XCD) + blockIdx.x / N_XCD >= (n_tiles + N_XCD - 1) / N_XCD) {
            return;
        }
        const uint32_t t = crowded_tile(turn, n_tiles);
        if (t == 0xFFFFFFFFu) {
            continue;
        }
        const Tile tile = args.tiles[t];
        const uint32_t first_tile = crowded_first_tile(args, tile);
        const CrowdedCell cell = args.cells[first_tile];
        const uint32_t n = uniform(cell.candidates);
        const uint32_t n_i = tile.count;
        const uint32_t n_units = (n + WAVE - 1) / WAVE;
        const bool tile_wrapped = (tile.wrapped & 1u) != 0;
        __syncthreads(); // (the tile before is done with the LDS)
        if (wave == 0) {
            bool out_of_range = false;
            SortedPoint point = {0.0, 0.0, 0.0, 0u, 0u};
            int32_t wx = 0, wy = 0, wz = 0;
            if (static_cast<uint32_t>(lane) < n_i) {
                const uint32_t at = tile.first + lane;
                point = args.sorted.p[at];
                wx = args.sorted.wx[at];
                wy = args.sorted.wy[at];
                wz = args.sorted.wz[at];
                sh.tile_index[lane] = point.index;
                sh.tile_x[lane] = point.x;
                sh.tile_y[lane] = point.y;
                sh.tile_z[lane] = point.z;
                sh.tile_wx[lane] = wx;
                sh.tile_wy[lane] = wy;
                sh.tile_wz[lane] = wz;
                out_of_range = beyond(wx, wy, wz, ORDERED_SHIFT_LIMIT);
                sh.rows[lane] = 0;
            }
            prepare_tile_tests(sh.tests, g, lane, n_i, point.x, point.y, point.z, wx, wy, wz, args.double_only);
            if (args.report != 0 && lane == 0 && sh.tests.usable == 0) {
                atomicAdd(&args.status->in_double, 1u);
            }
            if (__ballot(out_of_range) != 0 && lane == 0) {
                atomicOr(&args.status->unsuitable, 1u);
            }
        }
        __syncthreads();

        const CrowdedCandidate* candidates = args.candidates + static_cast<size_t>(cell.first_candidate) * WAVE;
        uint32_t* columns = args.columns + (static_cast<size_t>(cell.first_column) + static_cast<size_t>(t - first_tile) * n_units) * WAVE;
        uint32_t own_rows = 0;
        const bool single = uniform(sh.tests.usable) != 0;
        uint32_t unit = wave;
        for (; single && unit + (R - 1) * CROWDED_WAVES < n_units; unit += R * CROWDED_WAVES) {
            crowded_count_units<R, FULL>(sh, args.sorted, g, candidates, columns, unit, n, tile.first, n_i, lane, own_rows);
        }
        for (; single && unit < n_units; unit += CROWDED_WAVES) {
            crowded_count_units<1, FULL>(sh, args.sorted, g, candidates, columns, unit, n, tile.first, n_i, lane, own_rows);
        }
        for (uint32_t unit0 = wave * R; !single && unit0 < n_units; unit0 += CROWDED_WAVES * R) {
            SweepCandidates<R> c;
            uint32_t original[R], column[R];
            int32_t bx[R], by[R], bz[R];
            bool any_shift = false;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint32_t k = (unit0 + r) * WAVE + lane;
                c.x[r] = c.y[r] = c.z[r] = __builtin_nan("");
                c.tx[r] = c.ty[r] = c.tz[r] = 0.0;
                c.shift[r] = 0;
                c.position[r] = 0xFFFFFFFFu;
                column[r] = 0;
                original[r] = 0xFFFFFFFFu;
                bx[r] = by[r] = bz[r] = 0;
                if (k < n) {
                    const CrowdedCandidate candidate = candidates[k];
                    const SortedPoint point = args.sorted.p[candidate.at];
                    c.x[r] = point.x;
                    c.y[r] = point.y;
                    c.z[r] = point.z;
                    original[r] = point.index;
                    bx[r] = static_cast<int32_t>((candidate.biased >> 20) & 0x3ffu) - 512;
                    by[r] = static_cast<int32_t>((candidate.biased >> 10) & 0x3ffu) - 512;
                    bz[r] = static_cast<int32_t>(candidate.biased & 0x3ffu) - 512;
                    // a point is no neighbour of itself; a half list keeps a point with its own image under the rule of
                    // the reference (in a tile without wrapped points the shift of such a pair is the cell shift)
                    const bool never_with_itself =
                        (bx[r] | by[r] | bz[r]) == 0 || (!FULL && !half_keeps_self_image(bx[r], by[r], bz[r]));
                    c.position[r] = never_with_itself ? candidate.at : 0xFFFFFFFFu;
                }
                any_shift = any_shift || __ballot((bx[r] | by[r] | bz[r]) != 0) != 0;
            }
            if (!tile_wrapped) {
                if (any_shift) {
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        shift_vector(g, bx[r], by[r], bz[r], c.tx[r], c.ty[r], c.tz[r]);
                    }
                    sweep_and_count<R, true, FULL>(sh, tile.first, n_i, c, g.cutoff2, original, lane, column, own_rows);
                } else {
                    sweep_and_count<R, false, FULL>(sh, tile.first, n_i, c, g.cutoff2, original, lane, column, own_rows);
                }
            } else {
                // some points of the tile were moved into the box: the shift differs from point to point
                for (uint32_t p = 0; p < n_i; p++) {
                    const double xi = sh.tile_x[p];
                    const double yi = sh.tile_y[p];
                    const double zi = sh.tile_z[p];
                    const uint32_t index_i = sh.tile_index[p];
                    uint32_t found = 0;
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const int32_t sx = bx[r] + sh.tile_wx[p];
                        const int32_t sy = by[r] + sh.tile_wy[p];
                        const int32_t sz = bz[r] + sh.tile_wz[p];
                        double tx, ty, tz;
                        shift_vector(g, sx, sy, sz, tx, ty, tz);
                        const double vx = (c.x[r] - xi) + tx;
                        const double vy = (c.y[r] - yi) + ty;
                        const double vz = (c.z[r] - zi) + tz;
                        const double d2 = vx * vx + vy * vy + vz * vz;
                        const bool itself = index_i == original[r];
                        bool keep = d2 < g.cutoff2 && !(itself && (sx | sy | sz) == 0);
                        if (!FULL) {
                            keep = keep && (index_i < original[r] || (itself && half_keeps_self_image(sx, sy, sz)));
                        }
                        const uint64_t mask = __ballot(keep);
                        found += __popcll(mask);
                        column[r] = shift_in(column[r], mask);
                    }
                    if (static_cast<uint32_t>(lane) == p) {
                        own_rows += found;
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (unit0 + r < n_units) {
                    columns[(unit0 + r) * WAVE + lane] = column[r];
                }
            }
        }
        if (static_cast<uint32_t>(lane) < n_i && own_rows != 0) {
            atomicAdd(&sh.rows[lane], own_rows);
        }
        __syncthreads();
        if (threadIdx.x < n_i) {
            args.rows_of_point[sh.tile_index[threadIdx.x]] = sh.rows[threadIdx.x];
        }
    }
}

__global__ void publish_crowded_status(
    const CrowdedStatus* found, const uint64_t* total, const DeviceStatus* status, const uint64_t* cell_scan_end,
    CrowdedHostStatus* host
) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        host->found = *found;
        host->total_rows = total != nullptr ? *total : 0;
        host->first_bad_coordinate = status->first_bad_coordinate;
        host->n_tiles = static_cast<unsigned int>(*cell_scan_end >> 32);
    }
}

__global__ void clear_crowded_status(CrowdedStatus* status) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        *status = CrowdedStatus{};
    }
}

// ---------------------------------------------------------------------------------------------------------------
// WRITE: only the candidates with a hit go through the chunks (clusters of 500,000 points, P d, 700 -> 615 us; 200,000
// points, 55 per cell, half P S d D 440 -> 345 us).

template <bool STAGED, TileStores STORES>
__global__ __launch_bounds__(TILE_BLOCK, STAGED ? 4 : 5) void crowded_write_kernel(CrowdedArgs args, GridParams g) {
    __shared__ TileWriteShared<STAGED> sh;
    __shared__ uint32_t hits_of[4 * TILE_WAVES];
    __shared__ uint32_t beyond_chunk;
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    const uint32_t wave = uniform(threadIdx.x / WAVE);
    const CrowdedStatus found = *args.status;
    if (found.overflow != 0 || found.unsuitable != 0 || found.max_candidates > CROWDED_LARGE ||
        args.first_row[g.n_points] > args.capacity) {
        return;
    }
    const uint32_t n_tiles = static_cast<uint32_t>(args.cell_scan[g.n_cells] >> 32);
    for (uint32_t turn = 0;; turn++) {
        if (turn * (gridDim.x / N_XCD) + blockIdx.x / N_XCD >= (n_tiles + N_XCD - 1) / N_XCD) {
            return;
        }
        const uint32_t t = crowded_tile(turn, n_tiles);
        if (t == 0xFFFFFFFFu) {
            continue;
        }
        const Tile tile = args.tiles[t];
        const uint32_t first_tile = crowded_first_tile(args, tile);
        const CrowdedCell cell = args.cells[first_tile];
        const uint32_t n = uniform(cell.candidates);
        const uint32_t n_i = uniform(tile.count);
        const uint32_t n_units = (n + WAVE - 1) / WAVE;
        __syncthreads(); // (the tile before is done with the LDS)
        const bool moved = load_tile(sh, args.sorted, tile.first, n_i, args.first_row);
        const CrowdedCandidate* candidates = args.candidates + static_cast<size_t>(cell.first_candidate) * WAVE;
        const uint32_t* columns =
            args.columns + (static_cast<size_t>(cell.first_column) + static_cast<size_t>(t - first_tile) * n_units) * WAVE;
        // The candidates that some point of the tile has for a neighbour (about two thirds), TILE_CHUNK of them at a time: each
        // thread looks at one in TILE_BLOCK of the next 4 TILE_BLOCK candidates.
        constexpr uint32_t LOOK = 4;
        for (uint32_t first = 0; first < n;) {
            if (first != 0) {
                __syncthreads();
            }
            uint32_t column[LOOK];
            CrowdedCandidate candidate[LOOK];
            uint64_t mask[LOOK];
#pragma unroll
            for (uint32_t u = 0; u < LOOK; u++) {
                const uint32_t k = first + u * TILE_BLOCK + threadIdx.x;
                column[u] = 0;
                if (k < n) {
                    column[u] = columns[k];
                    candidate[u] = candidates[k];
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < LOOK; u++) {
                mask[u] = __ballot(column[u] != 0);
                if (lane == 0) {
                    hits_of[u * TILE_WAVES + wave] = __popcll(mask[u]);
                }
            }
            __syncthreads();
            uint32_t found = 0;
            uint32_t next = min(first + LOOK * TILE_BLOCK, n);
            bool shifted = moved;
#pragma unroll
            for (uint32_t u = 0; u < LOOK; u++) {
                uint32_t slot = found + rank_in_mask(mask[u]);
#pragma unroll
                for (uint32_t w = 0; w < TILE_WAVES; w++) {
                    const uint32_t hits = uniform(hits_of[u * TILE_WAVES + w]);
                    slot += w < wave ? hits : 0u;
                    found += hits;
                }
                const uint32_t k = first + u * TILE_BLOCK + threadIdx.x;
                if (column[u] != 0 && slot < TILE_CHUNK) {
                    const SortedPoint point = args.sorted.p[candidate[u].at];
                    sh.x[slot] = point.x;
                    sh.y[slot] = point.y;
                    sh.z[slot] = point.z;
                    sh.index[slot] = point.index;
                    sh.biased[slot] = candidate[u].biased;
                    sh.column[slot] = column[u];
                    shifted = shifted || candidate[u].biased != NO_SHIFT;
                }
                if (column[u] != 0 && slot == TILE_CHUNK) {
                    beyond_chunk = k; // the first that did not fit
                }
            }
            const uint32_t in_chunk = min(found, TILE_CHUNK);
            const uint32_t units_here = (in_chunk + WAVE - 1) / WAVE;
            // (the columns of the last unit beyond the last candidate)
            if (threadIdx.x < units_here * WAVE - in_chunk) {
                sh.column[in_chunk + threadIdx.x] = 0;
            }
            const bool any_shifted = __syncthreads_or(shifted) != 0;
            if (found > TILE_CHUNK) {
                next = uniform(beyond_chunk);
            }
            const bool more_chunks = first != 0 || next < n;
            first = next;
            if (in_chunk == 0) {
                continue;
            }
            if (any_shifted) {
                write_tile_chunk<true, STAGED, STORES>(sh, wave, g, args.out, n_i, units_here, more_chunks, lane);
            } else {
                write_tile_chunk<false, STAGED, STORES>(sh, wave, g, args.out, n_i, units_here, more_chunks, lane);
            }
        }
    }
}

} // namespace vesin_hip

#endif
