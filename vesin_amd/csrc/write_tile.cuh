// The writing pass of the in-order searches (ordered.cuh, crowded.cuh): what a workgroup does with a tile once the
// candidates of the tile's cell, in final order, and their hit columns are known.
//
// The workgroup brings TILE_CHUNK candidates at a time to LDS: coordinates, original index, shift, hit column. Its waves
// share the tile's points, in the order of their original indices. A wave holds the columns of the chunk in registers
// (lane l of unit u: candidate 64 u + l); for a point, the lanes whose column has the point's bit line up in LDS behind
// the rows of the points before it, as 16-bit entries (point, candidate), and entries that are consecutive rows of the
// list are then stored 64 at a time from multiples of 64 rows (whole cache lines in every output array). A step needs nothing from memory, and the shift
// vectors are only computed where some candidate of the chunk or point of the tile has a shift.
#ifndef VESIN_HIP_WRITE_TILE_CUH
#define VESIN_HIP_WRITE_TILE_CUH

#include "search.cuh"

namespace vesin_hip {

// LDS is what bounds the workgroups per compute unit: 31 KB, five of them (37 KB and four with vectors lined up).
constexpr int TILE_WAVES = 4;
constexpr int TILE_BLOCK = TILE_WAVES * WAVE;
constexpr uint32_t TILE_CHUNK = 704;
constexpr uint32_t TILE_UNITS = TILE_CHUNK / WAVE;
constexpr uint32_t TILE_STAGED = TILE_CHUNK + WAVE; // entries a wave lines up: one point's behind what a store left over
constexpr uint32_t NO_SHIFT = (512u << 20) | (512u << 10) | 512u; // biased
static_assert(TILE_CHUNK <= 1024 && TILE_POINTS <= 32, "an entry is (number of the point << 10) | number of the candidate");
static_assert(TILE_CHUNK * sizeof(uint32_t) <= TILE_WAVES * (TILE_STAGED + WAVE) * sizeof(uint16_t), "the columns share the entries' room");

/// STAGED: with room to line up the vectors of 64 rows per wave (the kernels of calls that return vectors).
template <bool STAGED>
struct TileWriteShared {
    double x[TILE_CHUNK], y[TILE_CHUNK], z[TILE_CHUNK];
    uint32_t index[TILE_CHUNK];
    uint32_t biased[TILE_CHUNK]; // biased shift, without the wrap of the first point
    __attribute__((aligned(16))) double vector_stage[TILE_WAVES][STAGED ? 3 * WAVE : 2];
    union {
        uint16_t staged[TILE_WAVES][TILE_STAGED + WAVE]; // (the last 64: where lanes without an entry write)
        uint32_t column[TILE_CHUNK]; // until every wave has them in its registers
    };
    double tile_x[TILE_POINTS], tile_y[TILE_POINTS], tile_z[TILE_POINTS];
    uint64_t tile_row[TILE_POINTS];  // first output row of each point that is not written yet
    uint32_t tile_rows[TILE_POINTS]; // rows of each point
    uint32_t tile_index[TILE_POINTS];
    uint32_t tile_wrap[TILE_POINTS]; // the three wraps in the fields of a biased shift
    uint32_t by_index[TILE_POINTS];  // the tile's points in the order of their original indices
};

/// The tile's points, by all threads of the workgroup; returns (in every thread) whether some point was moved into the
/// box by a box vector.
template <typename Shared>
__device__ __forceinline__ bool load_tile(
    Shared& sh, const SortedPoints& sorted, uint32_t first, uint32_t n_i, const uint64_t* __restrict__ first_row
) {
    bool moved = false;
    if (threadIdx.x < n_i) {
        const uint32_t at = first + threadIdx.x;
        const SortedPoint point = sorted.p[at];
        const int32_t wx = sorted.wx[at];
        const int32_t wy = sorted.wy[at];
        const int32_t wz = sorted.wz[at];
        sh.tile_index[threadIdx.x] = point.index;
        sh.tile_x[threadIdx.x] = point.x;
        sh.tile_y[threadIdx.x] = point.y;
        sh.tile_z[threadIdx.x] = point.z;
        // every field of biased shift and wrap together stays inside its ten bits (operands within +-255)
        sh.tile_wrap[threadIdx.x] =
            (static_cast<uint32_t>(wx) << 20) + (static_cast<uint32_t>(wy) << 10) + static_cast<uint32_t>(wz);
        const uint64_t row = first_row[point.index];
        sh.tile_row[threadIdx.x] = row;
        sh.tile_rows[threadIdx.x] = static_cast<uint32_t>(first_row[point.index + 1] - row);
        moved = (wx | wy | wz) != 0;
    }
    const bool any_moved = __syncthreads_or(moved) != 0;
    if (threadIdx.x < n_i) {
        const uint32_t own = sh.tile_index[threadIdx.x];
        uint32_t smaller = 0;
        for (uint32_t other = 0; other < n_i; other++) {
            smaller += sh.tile_index[other] < own ? 1u : 0u;
        }
        sh.by_index[smaller] = threadIdx.x;
    }
    return any_moved;
}

/// Stores the first `count` rows lined up by this wave as the rows `first_row` ... of the list. `zero`: the shift vector
/// of no shift, which is (+-0, +-0, +-0).
template <bool SHIFTED, bool STAGED, typename Shared>
__device__ __forceinline__ void store_tile_rows(
    Shared& sh, uint32_t wave, const GridParams& g, const SearchOutputs& out, const double (&zero)[3], uint32_t count,
    uint64_t first_row, uint32_t lane
) {
    const uint32_t skew = static_cast<uint32_t>(first_row % WAVE);
    const uint64_t aligned_row = uniform(first_row - skew);
    char* pairs = reinterpret_cast<char*>(out.pairs) + aligned_row * 16 + lane * 16u;
    char* shifts = reinterpret_cast<char*>(out.shifts) + aligned_row * 12 + lane * 12u;
    char* distances = reinterpret_cast<char*>(out.distances) + aligned_row * 8 + lane * 8u;
    for (uint32_t e0 = 0; e0 < count + skew; e0 += WAVE) {
        const uint32_t e = e0 + lane - skew;
        const bool active = e < count; // (not before the first row either: unsigned)
        const uint32_t entry = sh.staged[wave][active ? e : 0u];
        const uint32_t point = entry >> 10;
        const uint32_t candidate = entry & 1023u;
        double vx = sh.x[candidate] - sh.tile_x[point];
        double vy = sh.y[candidate] - sh.tile_y[point];
        double vz = sh.z[candidate] - sh.tile_z[point];
        const PairRow pair = {sh.tile_index[point], sh.index[candidate]};
        ShiftRow shift = {0, 0, 0};
        if (SHIFTED) {
            const uint32_t biased = sh.biased[candidate] + sh.tile_wrap[point];
            const int32_t sx = static_cast<int32_t>((biased >> 20) & 0x3ffu) - 512;
            const int32_t sy = static_cast<int32_t>((biased >> 10) & 0x3ffu) - 512;
            const int32_t sz = static_cast<int32_t>(biased & 0x3ffu) - 512;
            double tx, ty, tz;
            shift_vector(g, sx, sy, sz, tx, ty, tz);
            vx += tx;
            vy += ty;
            vz += tz;
            shift = ShiftRow{sx, sy, sz};
        } else {
            vx += zero[0];
            vy += zero[1];
            vz += zero[2];
        }
        if (active) {
            stream_store(pairs, pair);
            if (out.shifts != nullptr) {
                stream_store(shifts, shift);
            }
            if (out.distances != nullptr) {
                stream_store(distances, sqrt(vx * vx + vy * vy + vz * vz));
            }
        }
        if constexpr (STAGED) {
            store_vector_block(
                sh.vector_stage[wave], reinterpret_cast<char*>(out.vectors) + (aligned_row + e0) * 24, e0 == 0 ? skew : 0u,
                min(count + skew - e0, static_cast<uint32_t>(WAVE)), active, lane, vx, vy, vz
            );
        }
        pairs += 16 * WAVE;
        shifts += 12 * WAVE;
        distances += 8 * WAVE;
    }
}

/// The rows of this wave's share of the points with the candidates of the chunk in LDS. `more_chunks`: there are others.
template <bool SHIFTED, bool STAGED, typename Shared>
__device__ __forceinline__ void write_tile_chunk(
    Shared& sh, uint32_t wave, const GridParams& g, const SearchOutputs& out, uint32_t n_i, uint32_t units_here, bool more_chunks,
    uint32_t lane
) {
    double zero[3];
    shift_vector(g, 0, 0, 0, zero[0], zero[1], zero[2]);
    uint32_t column[TILE_UNITS];
#pragma unroll
    for (uint32_t u = 0; u < TILE_UNITS; u++) {
        column[u] = u < units_here ? sh.column[u * WAVE + lane] : 0u;
    }
    __syncthreads();
    const uint32_t per_wave = (n_i + TILE_WAVES - 1) / TILE_WAVES;
    const uint32_t turn_end = min(n_i, (wave + 1) * per_wave);
    uint32_t staged = 0;
    uint64_t staged_row = 0; // row of the first one lined up
    for (uint32_t turn = wave * per_wave;; turn++) {
        const bool more = turn < turn_end;
        const uint32_t p = uniform(sh.by_index[more ? turn : 0u]);
        const uint64_t row_p = uniform(sh.tile_row[p]);
        // (the rows of points with consecutive indices are consecutive rows of the list, as long as the candidates come
        // in one chunk)
        if (staged != 0 && (!more || row_p != staged_row + staged || staged + min(uniform(sh.tile_rows[p]), units_here * WAVE) > TILE_STAGED)) {
            wave_sync();
            store_tile_rows<SHIFTED, STAGED>(sh, wave, g, out, zero, staged, staged_row, lane);
            staged = 0;
            wave_sync();
        }
        if (!more) {
            break;
        }
        if (staged == 0) {
            staged_row = row_p;
        }
        const uint32_t bit = 1u << (n_i - 1 - p);
        const uint32_t entry = (p << 10) | lane;
        uint32_t rows_here = 0;
        // (no branches: the columns of units beyond the last are zero, and lanes without a hit write an entry that nobody
        // reads)
#pragma unroll
        for (uint32_t u = 0; u < TILE_UNITS; u++) {
            const bool hit = (column[u] & bit) != 0;
            const uint64_t mask = __ballot(hit);
            const uint32_t slot = __builtin_amdgcn_mbcnt_hi(
                static_cast<uint32_t>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), staged + rows_here)
            );
            sh.staged[wave][hit ? slot : TILE_STAGED + lane] = static_cast<uint16_t>(entry + u * WAVE);
            rows_here += __popcll(mask);
        }
        staged += rows_here;
        if (more_chunks) {
            wave_sync();
            if (lane == 0) {
                sh.tile_row[p] = row_p + rows_here;
            }
        }
    }
}

} // namespace vesin_hip

#endif
