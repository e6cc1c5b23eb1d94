// Gradient of the pair geometry with respect to points and box: the step that turns per-pair gradients of an
// energy model (dE/d distance, dE/d vector) into forces and virial. The reference does this with tensor
// operations (vesin-torch/src/vesin_torch.cpp:437-468): vectors_grad += distances_grad * vectors / distances;
// points_grad[j] += vectors_grad; points_grad[i] -= vectors_grad; box_grad = shifts^T . vectors_grad.
// Here it is one pass over the rows, 92 bytes read per pair; the sums are gathered per workgroup in LDS and go
// to memory with one fp64 atomic per point, component and workgroup.
#ifndef VESIN_HIP_BACKWARD_CUH
#define VESIN_HIP_BACKWARD_CUH

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

#include "device_common.cuh"
#include "policy.hpp"

namespace vesin_hip {

// Bound by reading the rows (56 bytes with a gradient of the distances only, 92 with everything). The table of sums fills
// 58 KB of LDS, so two workgroups share a compute unit: with 256 threads each, too few loads are in flight, with 1024
// the waves wait for each other where the table is filled and emptied (89 M rows, gradient of the distances: 1484 /
// 1056 / 1115 us with 256 / 512 / 1024 threads).
//
// Runs of one first point are summed without the LDS (shuffles do go through it), and all loads of a row are issued before
// its indices are looked at: 89 M rows, gradient of the distances, whole calls by the order of the list, unsorted 1436 -> 1334
// (sums) -> 1268 us (loads), sorted 1144 -> 1056 -> 963; the reads alone take 810 and 890 us. Reading the next rows ahead
// gives nothing on top (1274, 975), fewer bytes do not help any more (distances computed again from the vectors: the same),
// nor do 1024 threads or half the table for a third workgroup (5 to 25 % slower).
constexpr int BACKWARD_THREADS = 512;
static_assert(BACKWARD_ROWS % BACKWARD_THREADS == 0 && BACKWARD_STEP % BACKWARD_THREADS == 0, "whole rounds of the threads");

struct BackwardArgs {
    const size_t (*pairs)[2];
    const int32_t (*shifts)[3];    // nullptr: no gradient for the box
    const double* distances;
    const double (*vectors)[3];
    const double* distances_grad;  // nullptr: zero
    const double (*vectors_grad)[3]; // nullptr: zero
    size_t n_pairs;
    size_t n_points;
    double* points_grad;           // [n_points][3] or nullptr
    double* box_grad;              // [3][3] or nullptr
    uint32_t* bad_index;           // set to 1 when a pair names a point that does not exist
    size_t rows_per_block;         // a multiple of BACKWARD_THREADS (backward_rows_per_block, policy.hpp)
};

/// Sum over the 64 lanes of a wave, result in every lane.
__device__ inline double wave_sum(double value) {
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        value += __shfl_xor(value, offset, WAVE);
    }
    return value;
}

/// One step of a sum over runs: adds what the lane `CTRL` names (a DPP control, for the rows of `ROW_MASK`) holds, where that
/// lane belongs to the same run.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double add_from(double value, bool same_run) {
    const uint64_t there = dpp_or_zero64<CTRL, ROW_MASK>(static_cast<uint64_t>(__double_as_longlong(value)));
    return value + (same_run ? __longlong_as_double(static_cast<long long>(there)) : 0.0);
}

/// Sums a run of lanes that name the same point into the last lane of the run. `heads` has one bit per lane that starts a
/// run. (Data moves with DPP only: with shuffles, which go through the LDS that the table is in, see pairs_backward_kernel.)
__device__ inline void sum_runs(uint64_t heads, double& gx, double& gy, double& gz) {
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    const uint64_t up_to_here = heads & (~0ull >> (63 - lane));
    const uint32_t start = 63u - static_cast<uint32_t>(__builtin_clzll(up_to_here)); // (lane 0 starts a run)
    auto step = [&](auto control, auto row_mask, bool same_run) {
        constexpr int CTRL = decltype(control)::value;
        constexpr int ROW_MASK = decltype(row_mask)::value;
        gx = add_from<CTRL, ROW_MASK>(gx, same_run);
        gy = add_from<CTRL, ROW_MASK>(gy, same_run);
        gz = add_from<CTRL, ROW_MASK>(gz, same_run);
    };
    const uint32_t in_row = lane % 16;
    step(std::integral_constant<int, 0x111>(), std::integral_constant<int, 0xf>(), in_row >= 1 && start + 1 <= lane);
    step(std::integral_constant<int, 0x112>(), std::integral_constant<int, 0xf>(), in_row >= 2 && start + 2 <= lane);
    step(std::integral_constant<int, 0x114>(), std::integral_constant<int, 0xf>(), in_row >= 4 && start + 4 <= lane);
    step(std::integral_constant<int, 0x118>(), std::integral_constant<int, 0xf>(), in_row >= 8 && start + 8 <= lane);
    step(std::integral_constant<int, 0x142>(), std::integral_constant<int, 0xa>(), lane / 16 % 2 == 1 && start < lane - in_row);
    step(std::integral_constant<int, 0x143>(), std::integral_constant<int, 0xc>(), lane >= 32 && start < 32);
}

/// Sums of one workgroup, by point, in LDS: rows that follow each other in a list name few different points (the
/// points of a few cells), so most additions meet here and only one sum per point and workgroup goes to memory,
/// where an atomic on a line shared by all compute dies costs far more than one in LDS.
///
/// The table is open addressing in groups of eight slots: the eight points 8k ... 8k + 7 share a group, each at its own
/// place in it. Points of neighbouring indices are then neighbours in the table, and the workgroup's atomics to
/// memory, one lane per component, come as stretches of up to 192 consecutive bytes. (Measured with 512 threads, 89 M
/// rows, gradient of the distances, points spread by a hash of the whole index and added one point per lane -> like
/// this: 1358 -> 1057 us, sorted 1785 -> 1101 us, atoms in no order 1333 -> 1195 us: 4.7 TB/s of rows read, where a
/// plain copy on this GPU moves 4.8.)
constexpr uint32_t BACKWARD_SLOTS = 2048;
constexpr uint32_t BACKWARD_GROUP = 8;
constexpr uint32_t BACKWARD_PROBES = 8;
constexpr uint32_t BACKWARD_EMPTY = 0xFFFFFFFFu;

struct BackwardShared {
    uint32_t keys[BACKWARD_SLOTS];
    double sums[BACKWARD_SLOTS][3];
    double box[BACKWARD_THREADS / WAVE][9];
};

__device__ inline void add_to_point(BackwardShared& shared, double* points_grad, size_t point, double gx, double gy, double gz) {
    const uint32_t key = static_cast<uint32_t>(point);
    uint32_t slot = (((key / BACKWARD_GROUP) * 2654435761u) >> (32 - 8)) * BACKWARD_GROUP + key % BACKWARD_GROUP;
    static_assert(BACKWARD_SLOTS == (1u << 8) * BACKWARD_GROUP, "the hash keeps 8 bits");
    for (uint32_t probe = 0; probe < BACKWARD_PROBES; probe++) {
        // most points are in the table already: a read, which all lanes with the same point share, comes before the
        // compare-and-swap, which goes through them one by one
        uint32_t found = __atomic_load_n(&shared.keys[slot], __ATOMIC_RELAXED);
        if (found == BACKWARD_EMPTY) {
            found = atomicCAS(&shared.keys[slot], BACKWARD_EMPTY, key);
        }
        if (found == BACKWARD_EMPTY || found == key) {
            unsafeAtomicAdd(&shared.sums[slot][0], gx);
            unsafeAtomicAdd(&shared.sums[slot][1], gy);
            unsafeAtomicAdd(&shared.sums[slot][2], gz);
            return;
        }
        slot = (slot + BACKWARD_GROUP) & (BACKWARD_SLOTS - 1);
    }
    // the neighbourhood of the slot is taken by other points
    unsafeAtomicAdd(points_grad + 3 * point + 0, gx);
    unsafeAtomicAdd(points_grad + 3 * point + 1, gy);
    unsafeAtomicAdd(points_grad + 3 * point + 2, gz);
}

__global__ __launch_bounds__(BACKWARD_THREADS) void pairs_backward_kernel(BackwardArgs args) {
    __shared__ BackwardShared shared;
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    double box_sum[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    bool any_shift = false;

    if (args.points_grad != nullptr) {
        for (uint32_t slot = threadIdx.x; slot < BACKWARD_SLOTS; slot += BACKWARD_THREADS) {
            shared.keys[slot] = BACKWARD_EMPTY;
            shared.sums[slot][0] = 0.0;
            shared.sums[slot][1] = 0.0;
            shared.sums[slot][2] = 0.0;
        }
        __syncthreads();
    }

    // a workgroup takes rows that follow each other; every lane of a wave runs the same number of rounds (the sums
    // over runs use the whole wave)
    const size_t block_first = static_cast<size_t>(blockIdx.x) * args.rows_per_block;
    const size_t block_end = min(block_first + args.rows_per_block, args.n_pairs);
    for (size_t base = block_first + (threadIdx.x & ~(WAVE - 1)); base < block_end; base += BACKWARD_THREADS) {
        const size_t row = base + lane;
        bool active = row < block_end;
        // rows that do not count carry an index no point has, so that they never join the run of a neighbour
        size_t i = ~size_t(0);
        size_t j = 0;
        double gx = 0.0, gy = 0.0, gz = 0.0;
        double dg = 0.0, d = 1.0, vx = 0.0, vy = 0.0, vz = 0.0;
        if (active) { // (all loads of the row, none of which waits for another)
            i = args.pairs[row][0];
            j = args.pairs[row][1];
            if (args.vectors_grad != nullptr) {
                gx = args.vectors_grad[row][0];
                gy = args.vectors_grad[row][1];
                gz = args.vectors_grad[row][2];
            }
            if (args.distances_grad != nullptr) {
                dg = args.distances_grad[row];
                d = args.distances[row];
                vx = args.vectors[row][0];
                vy = args.vectors[row][1];
                vz = args.vectors[row][2];
            }
            if (i >= args.n_points || j >= args.n_points) {
                *args.bad_index = 1;
                active = false;
                i = ~size_t(0);
            }
        }
        if (active) {
            if (args.distances_grad != nullptr) {
                gx += dg * vx / d;
                gy += dg * vy / d;
                gz += dg * vz / d;
            }
            if (args.shifts != nullptr) {
                const int32_t s0 = args.shifts[row][0];
                const int32_t s1 = args.shifts[row][1];
                const int32_t s2 = args.shifts[row][2];
                if ((s0 | s1 | s2) != 0) {
                    any_shift = true;
                    const double s[3] = {static_cast<double>(s0), static_cast<double>(s1), static_cast<double>(s2)};
#pragma unroll
                    for (int a = 0; a < 3; a++) {
                        box_sum[3 * a + 0] += s[a] * gx;
                        box_sum[3 * a + 1] += s[a] * gy;
                        box_sum[3 * a + 2] += s[a] * gz;
                    }
                }
            }
        }

        if (args.points_grad != nullptr) {
            if (active) {
                add_to_point(shared, args.points_grad, j, gx, gy, gz);
            }
            // rows of one first point often sit next to each other (always in a sorted list): one addition per run
            const size_t before = __shfl_up(static_cast<unsigned long long>(i), 1, WAVE);
            const bool head = lane == 0 || before != i;
            const uint64_t heads = __ballot(head);
            double mx = -gx;
            double my = -gy;
            double mz = -gz;
            bool add = active;
            if (__popcll(heads) <= 32) {
                sum_runs(heads, mx, my, mz);
                add = active && (lane == 63 || (heads >> (lane + 1) & 1u) != 0);
            }
            if (add) {
                add_to_point(shared, args.points_grad, i, mx, my, mz);
            }
        }
    }

    if (args.points_grad != nullptr) {
        __syncthreads();
        for (uint32_t at = threadIdx.x; at < 3 * BACKWARD_SLOTS; at += BACKWARD_THREADS) {
            const uint32_t slot = at / 3;
            const uint32_t key = shared.keys[slot];
            if (key != BACKWARD_EMPTY) {
                unsafeAtomicAdd(args.points_grad + 3 * static_cast<size_t>(key) + (at - 3 * slot), shared.sums[slot][at - 3 * slot]);
            }
        }
    }

    if (args.box_grad != nullptr) {
        // one atomic per workgroup and component: they all go to the same 72 bytes, one after the other (with one per
        // wave a list of 2.1 M rows took 150 us instead of 57, one of 89 M rows 1864 us instead of 1576)
        const uint32_t wave = threadIdx.x / WAVE;
        const bool wave_has_shift = __ballot(any_shift) != 0;
#pragma unroll
        for (int k = 0; k < 9; k++) {
            const double total = wave_has_shift ? wave_sum(box_sum[k]) : 0.0;
            if (lane == 0) {
                shared.box[wave][k] = total;
            }
        }
        __syncthreads();
        if (threadIdx.x < 9) {
            double total = 0.0;
            for (int w = 0; w < BACKWARD_THREADS / WAVE; w++) {
                total += shared.box[w][threadIdx.x];
            }
            if (total != 0.0) {
                unsafeAtomicAdd(args.box_grad + threadIdx.x, total);
            }
        }
    }
}

} // namespace vesin_hip

#endif
