// The writing pass of the in-order searches (ordered_tile.cuh, crowded.cuh): what a workgroup does with a tile once the
// candidates of the tile's cell, in final order, and their hit columns are known.
//
// The workgroup brings TILE_CHUNK candidates at a time to LDS: coordinates, original index, shift, hit column. The rows that
// they make are lined up in LDS, in the order of the tile's points by original index, as 16-bit entries (point, candidate)
// in a line of places that is common to the workgroup: where a point's rows start in it follows from its first row and its
// number of rows. Then its waves store 64 places at a time. A place knows its row by one addition (the difference is kept per
// point), so a step takes the end of one run of consecutive rows and the start of the next, and a run starts at a place that
// is its first row modulo TILE_GRANULE: steps cut runs between whole 64-byte pieces of every output array. Those two matter
// most here: a store occupies the compute unit's way to memory for all 64 lanes whether they have rows or not, and pieces
// that two stores share cost several times what whole ones do (1,000,000 atoms of diamond, P S d, stored run by run from
// multiples of 64 rows: 0.92 ms; with the incomplete pieces left out 0.70 ms). A step needs nothing from memory, and the
// shift vectors are only computed where some candidate of the chunk or point of the tile has a shift.
#ifndef VESIN_HIP_WRITE_TILE_CUH
#define VESIN_HIP_WRITE_TILE_CUH

#include "policy.hpp"
#include "search.cuh"

namespace vesin_hip {

// LDS and registers leave room for five workgroups per compute unit, four with vectors (six and five by spilling registers:
// 1,000,000 atoms of diamond, P S d, 1010 against 810 us).
constexpr int TILE_WAVES = 4;
constexpr int TILE_BLOCK = TILE_WAVES * WAVE;
constexpr uint32_t TILE_CHUNK = 512;
constexpr uint32_t TILE_UNITS = TILE_CHUNK / WAVE;
constexpr uint32_t TILE_LINE = 2560;        // places of the line of entries
constexpr uint32_t TILE_GRANULE = 16;       // rows: whole 64-byte pieces of pairs, shifts, distances and vectors
constexpr uint16_t NO_ENTRY = 0xFFFFu;
constexpr uint32_t NO_SHIFT = (512u << 20) | (512u << 10) | 512u; // biased
static_assert(TILE_CHUNK <= 1024 && TILE_POINTS <= 32, "an entry is (number of the point << 10) | number of the candidate");
static_assert(TILE_LINE % WAVE == 0 && TILE_CHUNK * sizeof(uint32_t) <= TILE_LINE * sizeof(uint16_t), "the columns share the entries' room");

/// STAGED: with room to line up the vectors of 64 rows per wave (the kernels of calls that return vectors).
template <bool STAGED>
struct TileWriteShared {
    double x[TILE_CHUNK], y[TILE_CHUNK], z[TILE_CHUNK];
    uint32_t index[TILE_CHUNK];
    uint32_t biased[TILE_CHUNK]; // biased shift, without the wrap of the first point
    __attribute__((aligned(16))) double vector_stage[TILE_WAVES][STAGED ? 3 * WAVE : 2];
    union {
        uint16_t entry[TILE_LINE + WAVE]; // (the last 64: where lanes without an entry write)
        uint32_t column[TILE_CHUNK]; // until every wave has them in its registers
    };
    double tile_x[TILE_POINTS], tile_y[TILE_POINTS], tile_z[TILE_POINTS];
    uint64_t tile_row[TILE_POINTS];  // first output row of each point that is not written yet
    uint32_t shared_granules[TILE_LINE / TILE_GRANULE / 32]; // a bit per granule of the line: some run starts or ends in it
    uint64_t row_of_place[TILE_POINTS]; // what a place in the line is off by from its row, per point
    uint32_t tile_rows[TILE_POINTS]; // rows of each point
    uint32_t first_place[TILE_POINTS], gap_before[TILE_POINTS]; // of each point in the line
    uint32_t chunk_rows[TILE_POINTS]; // and those of the chunk, when there are several
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

/// The top bits of the lanes' columns, which are shifted to the left: one vector instruction.
__device__ __forceinline__ uint64_t shift_out(uint32_t& column) {
    uint64_t carry;
    asm("v_add_co_u32_e64 %0, %1, %2, %2" : "=v"(column), "=s"(carry) : "v"(column));
    return carry;
}

/// Stores as TileStores (policy.hpp) says.
template <typename T>
__device__ __forceinline__ void cached_store(void* address, T value) {
    *reinterpret_cast<T*>(address) = value;
}

template <TileStores STORES, typename T>
__device__ __forceinline__ void store_row(void* address, T value) {
    if constexpr (STORES == STORE_CACHED) {
        cached_store(address, value);
    } else {
        stream_store(address, value);
    }
}

/// Stores the rows of the 64 places from `step` on (`first_place`: the number of the first place of the line in LDS). `zero`:
/// the shift vector of no shift, which is (+-0, +-0, +-0).
template <bool SHIFTED, bool STAGED, TileStores STORES, typename Shared>
__device__ __forceinline__ void store_tile_step(
    Shared& sh, uint32_t wave, const GridParams& g, const SearchOutputs& out, const double (&zero)[3], uint32_t first_place,
    uint32_t step, uint32_t lane
) {
    const uint32_t held = sh.entry[step + lane];
    const bool active = held != NO_ENTRY;
    const uint32_t entry = active ? held : 0u;
    const uint32_t point = entry >> 10;
    const uint32_t candidate = entry & 1023u;
    const uint64_t row = sh.row_of_place[point] + (first_place + step + lane);
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
    } else if (STAGED) { // (a distance is the same without it)
        vx += zero[0];
        vy += zero[1];
        vz += zero[2];
    }
    if constexpr (STORES == STORE_BY_GRANULE) {
        // (a bit per granule of the step)
        const uint32_t cached = uniform(sh.shared_granules[step / (32 * TILE_GRANULE)]) >> (step / TILE_GRANULE % 32) & 0xFu;
        const bool streamed = (cached >> (lane / TILE_GRANULE) & 1u) == 0;
        const double distance = out.distances != nullptr ? sqrt(vx * vx + vy * vy + vz * vz) : 0.0;
        if (active && streamed) {
            stream_store(out.pairs + 2 * row, pair);
            if (out.shifts != nullptr) {
                stream_store(out.shifts + 3 * row, shift);
            }
            if (out.distances != nullptr) {
                stream_store(out.distances + row, distance);
            }
        }
        if (cached != 0) {
            if (active && !streamed) {
                cached_store(out.pairs + 2 * row, pair);
                if (out.shifts != nullptr) {
                    cached_store(out.shifts + 3 * row, shift);
                }
                if (out.distances != nullptr) {
                    cached_store(out.distances + row, distance);
                }
            }
        }
    } else if (active) {
        store_row<STORES>(out.pairs + 2 * row, pair);
        if (out.shifts != nullptr) {
            store_row<STORES>(out.shifts + 3 * row, shift);
        }
        if (out.distances != nullptr) {
            store_row<STORES>(out.distances + row, sqrt(vx * vx + vy * vy + vz * vz));
        }
    }
    if constexpr (STAGED) {
        // The vectors as 16-byte pieces of consecutive addresses (see store_vector_block): two components of one row, or of
        // two rows next to each other in the line, which are next to each other in the list when they are off by the same.
        double* stage = sh.vector_stage[wave];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        stage[3 * lane + 0] = vx;
        stage[3 * lane + 1] = vy;
        stage[3 * lane + 2] = vz;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (uint32_t turn = 0; turn < 2; turn++) {
            const uint32_t piece = turn * WAVE + lane; // 96 pieces of 16 bytes make 64 rows
            if (piece < 3 * WAVE / 2) {
                const uint32_t first = 2 * piece / 3;
                const uint32_t second = (2 * piece + 1) / 3;
                const uint32_t first_entry = sh.entry[step + first];
                const uint32_t second_entry = sh.entry[step + second];
                const bool first_there = first_entry != NO_ENTRY;
                const bool second_there = second_entry != NO_ENTRY;
                const uint64_t first_off = sh.row_of_place[(first_there ? first_entry : 0u) >> 10];
                const uint64_t second_off = sh.row_of_place[(second_there ? second_entry : 0u) >> 10];
                const VectorHead two = {stage[2 * piece], stage[2 * piece + 1]};
                double* target = out.vectors + 3 * (first_off + (first_place + step)) + 2 * piece;
                if (first_there && second_there && first_off == second_off) {
                    store_row<STORES>(target, two);
                } else {
                    if (first_there) {
                        store_row<STORES>(target, two.x);
                    }
                    if (second_there) {
                        store_row<STORES>(out.vectors + 3 * (second_off + (first_place + step)) + 2 * piece + 1, two.y);
                    }
                }
            }
        }
    }
}

/// The rows that the candidates of the chunk in LDS make, by all waves of the workgroup. `more_chunks`: there are others.
template <bool SHIFTED, bool STAGED, TileStores STORES, typename Shared>
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
    // The points of this wave: their bits, moved to the top of the columns, come out one after the other as the carries of
    // column + column, which are the masks of the lanes with a hit.
    const uint32_t per_wave = (n_i + TILE_WAVES - 1) / TILE_WAVES;
    const uint32_t first_point = wave * per_wave;
    const uint32_t end_point = min(n_i, first_point + per_wave);
    uint32_t shifted_out[TILE_UNITS];
    auto move_to_top = [&]() {
#pragma unroll
        for (uint32_t u = 0; u < TILE_UNITS; u++) {
            shifted_out[u] = column[u] << ((32u - n_i + first_point) % 32u);
        }
    };
    move_to_top();
    if (more_chunks) {
        for (uint32_t p = first_point; p < end_point; p++) {
            uint32_t rows = 0;
#pragma unroll
            for (uint32_t u = 0; u < TILE_UNITS; u++) {
                rows += __popcll(shift_out(shifted_out[u]));
            }
            if (lane == 0) {
                sh.chunk_rows[p] = rows;
            }
        }
        move_to_top();
    }
    __syncthreads();

    // Where the rows of the points go in the line: behind those of the point before, after a gap where that brings the place
    // to the first row modulo TILE_GRANULE (none when the rows are consecutive rows of the list). Lane t: the point that
    // comes t-th by original index; every wave for itself.
    uint32_t place = 0, gap = 0, rows = 0;
    uint64_t row = 0;
    bool starts = false; // a run
    if (lane < n_i) {
        const uint32_t p = sh.by_index[lane];
        row = sh.tile_row[p];
        rows = more_chunks ? sh.chunk_rows[p] : sh.tile_rows[p];
    }
    {
        const uint32_t rows_before = static_cast<uint32_t>(__shfl_up(static_cast<int>(rows), 1));
        const uint64_t end_before = __shfl_up(static_cast<unsigned long long>(row + rows), 1);
        starts = lane < n_i && (lane == 0 || row != end_before);
        gap = (static_cast<uint32_t>(row) - (lane == 0 ? 0u : static_cast<uint32_t>(end_before))) % TILE_GRANULE;
        place = wave_inclusive_scan(gap + (lane == 0 ? 0u : rows_before));
        if (lane < n_i) {
            // (the same from every wave, which only needs what it wrote itself before the next barrier)
            const uint32_t p = sh.by_index[lane];
            sh.row_of_place[p] = row - place;
            sh.first_place[p] = place;
            sh.gap_before[p] = gap;
        }
    }
    wave_sync();
    const uint32_t end = read_lane(place + rows, static_cast<int>(n_i - 1));
    for (uint32_t first_place = 0; first_place < end; first_place += TILE_LINE) {
        if (first_place != 0) {
            __syncthreads(); // (the line before is stored)
        }
        if (STORES == STORE_BY_GRANULE && wave == 0) {
            if (lane < TILE_LINE / TILE_GRANULE / 32) {
                sh.shared_granules[lane] = 0;
            }
            wave_sync();
            auto mark = [&](uint32_t where) { // a run starts, or the one before has ended
                where -= first_place;
                if (where % TILE_GRANULE != 0 && where < TILE_LINE) {
                    atomicOr(&sh.shared_granules[where / (32 * TILE_GRANULE)], 1u << (where / TILE_GRANULE % 32));
                }
            };
            if (starts) {
                mark(place);
                mark(place - gap);
            }
            if (lane == n_i - 1) {
                mark(place + rows);
            }
        }
        if (first_place != 0) {
            move_to_top();
        }
        for (uint32_t p = first_point; p < end_point; p++) {
            // (places before this line are beyond it as well: unsigned)
            const uint32_t start = uniform(sh.first_place[p]) - first_place;
            const uint32_t before = uniform(sh.gap_before[p]);
            if (lane < before && start - 1 - lane < TILE_LINE) {
                sh.entry[start - 1 - lane] = NO_ENTRY;
            }
            const uint32_t entry = (p << 10) | lane;
            uint32_t next = start;
            // (no branches: the columns of units beyond the last are zero, and lanes without a hit write an entry that nobody
            // reads)
#pragma unroll
            for (uint32_t u = 0; u < TILE_UNITS; u++) {
                const uint64_t mask = shift_out(shifted_out[u]);
                const uint32_t slot = __builtin_amdgcn_mbcnt_hi(
                    static_cast<uint32_t>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), next)
                );
                const uint32_t wanted = __builtin_amdgcn_inverse_ballot_w64(mask) ? slot : 0xFFFFFFFFu;
                sh.entry[min(wanted, TILE_LINE + lane)] = static_cast<uint16_t>(entry + u * WAVE);
                next += __popcll(mask);
            }
        }
        if (wave == TILE_WAVES - 1 && end - first_place + lane < TILE_LINE) {
            sh.entry[end - first_place + lane] = NO_ENTRY; // (up to the end of the last step)
        }
        __syncthreads();
        const uint32_t places_here = min(end - first_place, TILE_LINE);
        for (uint32_t step = wave * WAVE; step < places_here; step += TILE_WAVES * WAVE) {
            store_tile_step<SHIFTED, STAGED, STORES>(sh, wave, g, out, zero, first_place, step, lane);
        }
    }
    if (more_chunks && wave == 0 && lane < n_i) {
        sh.tile_row[sh.by_index[lane]] = row + rows;
    }
}

} // namespace vesin_hip

#endif
