// Distance tests of a tile's points against its candidates in single precision, for the counting passes of the in-order
// searches: one lane per candidate and unit, six vector instructions per test (three products and sums, two comparisons,
// one shift into the hit column) where a test in double precision takes fourteen.
//
// Everything is taken relative to the tile's first point, in double precision, and rounded once: a = fl(A) for the points of
// the tile, c = fl(C) for the candidates, shifts and wraps included. With h = |c|^2 (rounded), the test is
//   t = -2 a.c + h  <  rc^2 -+ eps - |a|^2 :
// below the smaller bound the pair is within the cutoff, not below the larger one it is not, and whoever calls decides
// anything in between (and everything, when the tile is too wide for a useful eps) with the reference's own arithmetic in
// double precision. So the decisions are the reference's, bit for bit.
//
// The bound. u = 2^-24, s = the largest |A| of the tile, d the distance of the pair. Rounding a and c moves d^2 by at most
// 2 d u (|A| + |C|); h is off by 3 u |c|^2, the three sums of products by u (|c|^2 + 2 |a| |c|) each, the bounds by
// u (rc^2 + s^2) each. A pair whose distance is next to the cutoff has |C| <= s + rc: together
// u (14 s^2 + 22 s rc + 10 rc^2), to first order. Half as much again as twice that is eps (second orders, and what the
// square root and its sums lose). At other distances the error grows by less than the distance from the cutoff does, while
// eps is below a hundredth of rc^2, which is asked for. What double precision leaves in A and C and in the reference's own
// vectors is 2^-47 (|X| + s + rc + 512 |H|) at most, X the first point, |H| the sum of the absolute elements of the box,
// shifts within +-510.
#ifndef VESIN_HIP_TILE_TEST_CUH
#define VESIN_HIP_TILE_TEST_CUH

#include "fused.cuh"
#include "search.cuh"

namespace vesin_hip {

/// `values` with `value` in lane `where` (both the same in every lane): one vector instruction, where a comparison and a
/// selection take three. (The compiler has no builtin of its own for its intrinsic: the build tries its name first.)
#ifdef VESIN_HIP_NO_WRITE_LANE
__device__ __forceinline__ uint32_t with_lane(uint32_t values, uint32_t value, uint32_t where) {
    return static_cast<uint32_t>(lane_id()) == where ? value : values;
}
#else
extern "C" __device__ uint32_t vesin_write_lane(uint32_t value, uint32_t where, uint32_t values) __asm("llvm.amdgcn.writelane.i32");

__device__ __forceinline__ uint32_t with_lane(uint32_t values, uint32_t value, uint32_t where) {
    return vesin_write_lane(uniform(value), uniform(where), values);
}
#endif

struct TileTests {
    float4 point[TILE_POINTS]; // -2 a, lower bound
    float upper[TILE_POINTS];
    double origin[3];
    uint32_t usable;
};

/// By one wave, whose lane p < n_i holds point p of the tile: coordinates and the box vectors that it was moved by.
/// `double_only`: not zero: they are not used.
__device__ __forceinline__ void prepare_tile_tests(
    TileTests& tests, const GridParams& g, uint32_t lane, uint32_t n_i, double x, double y, double z, int32_t wx, int32_t wy, int32_t wz,
    uint32_t double_only
) {
    double tx, ty, tz;
    shift_vector(g, -wx, -wy, -wz, tx, ty, tz);
    x += tx;
    y += ty;
    z += tz;
    const double ox = __shfl(x, 0);
    const double oy = __shfl(y, 0);
    const double oz = __shfl(z, 0);
    const float ax = static_cast<float>(x - ox);
    const float ay = static_cast<float>(y - oy);
    const float az = static_cast<float>(z - oz);
    const double square = static_cast<double>(ax) * ax + static_cast<double>(ay) * ay + static_cast<double>(az) * az;
    double widest = lane < n_i ? square : 0.0;
#pragma unroll
    for (int offset = TILE_POINTS / 2; offset > 0; offset >>= 1) {
        widest = fmax(widest, __shfl_xor(widest, offset));
    }
    widest = __shfl(widest, 0);
    double box = 0.0;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        box += fabs(g.H[k]);
    }
    const double rc = sqrt(g.cutoff2);
    const double s = sqrt(widest);
    const double rounding = 0x1p-47 * (fabs(ox) + fabs(oy) + fabs(oz) + s + rc + 512.0 * box);
    const double eps = 3.0 * 0x1p-24 * (14.0 * widest + 22.0 * s * rc + 10.0 * g.cutoff2) + 8.0 * rc * rounding;
    if (lane < n_i) {
        tests.point[lane] = float4{-2.0f * ax, -2.0f * ay, -2.0f * az, static_cast<float>(g.cutoff2 - eps - square)};
        tests.upper[lane] = static_cast<float>(g.cutoff2 + eps - square);
    }
    if (lane == 0) {
        tests.origin[0] = ox;
        tests.origin[1] = oy;
        tests.origin[2] = oz;
        // (also not for cutoffs whose squares come near the range of single precision)
        tests.usable = double_only == 0 && eps < 0.01 * g.cutoff2 && g.cutoff2 > 1e-20 && g.cutoff2 < 1e+20 ? 1u : 0u;
    }
}

/// What a lane holds of R candidates.
template <int R>
struct TestCandidates {
    float x[R], y[R], z[R]; // relative to the origin of the tests; NOT_THERE for lanes without a candidate
    uint32_t limit[R];      // half lists: points of a smaller original index than this are partners
};

constexpr float NOT_THERE = 1.0e30f;

/// The tile's points against R units of candidates: hit columns (the first point in the highest bit used), lane p of `rows`
/// gets the hits of point p. Returns the lanes of pairs that are too close to the cutoff to call. A point's pair with
/// itself counts as one, unless the list is half and `limit` keeps it out.
template <int R, bool FULL>
__device__ __forceinline__ uint64_t test_tile(
    const TileTests& tests, const uint32_t* tile_index, uint32_t n_i, const TestCandidates<R>& c, uint32_t (&column)[R], uint32_t& rows
) {
    constexpr int AHEAD = 4; // points whose data is read at a time
    float square[R];
    uint64_t uncertain = 0;
    rows = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        square[r] = __builtin_fmaf(c.z[r], c.z[r], __builtin_fmaf(c.y[r], c.y[r], c.x[r] * c.x[r]));
        column[r] = 0;
    }
    auto test_points = [&](uint32_t first, auto number) {
        constexpr int N = decltype(number)::value;
        float4 point[N];
        float upper[N];
        uint32_t index[N];
#pragma unroll
        for (int k = 0; k < N; k++) {
            point[k] = tests.point[first + k];
            upper[k] = tests.upper[first + k];
            index[k] = FULL ? 0u : tile_index[first + k];
        }
#pragma unroll
        for (int k = 0; k < N; k++) {
            uint32_t found = 0;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float t =
                    __builtin_fmaf(point[k].x, c.x[r], __builtin_fmaf(point[k].y, c.y[r], __builtin_fmaf(point[k].z, c.z[r], square[r])));
                uint64_t within = __ballot(t < point[k].w);
                uint64_t perhaps = __ballot(t < upper[k]);
                if (!FULL) {
                    const uint64_t partners = __ballot(index[k] < c.limit[r]);
                    within &= partners;
                    perhaps &= partners;
                }
                uncertain |= perhaps & ~within;
                column[r] = shift_in(column[r], within);
                found += __popcll(within);
            }
            rows = with_lane(rows, found, first + k);
        }
    };
    uint32_t first = 0;
    for (; first + AHEAD <= n_i; first += AHEAD) {
        test_points(first, std::integral_constant<int, AHEAD>());
    }
    for (; first < n_i; first++) {
        test_points(first, std::integral_constant<int, 1>());
    }
    return uncertain;
}

/// The same pairs once more, where test_tile found some too close to the cutoff: those are decided by
/// `exact(r, p)` (whether the lane's candidate r is within the cutoff of point p, in double precision), the others as they
/// were.
template <int R, bool FULL, typename Exact>
__device__ __forceinline__ void resolve_tile(
    const TileTests& tests, const uint32_t* tile_index, uint32_t n_i, const TestCandidates<R>& c, uint32_t (&column)[R], uint32_t& rows,
    const Exact& exact
) {
    const uint32_t lane = static_cast<uint32_t>(lane_id());
    for (uint32_t p = 0; p < n_i; p++) {
        const float4 point = tests.point[p];
        const float upper = tests.upper[p];
        const uint32_t bit = 1u << (n_i - 1 - p);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float square = __builtin_fmaf(c.z[r], c.z[r], __builtin_fmaf(c.y[r], c.y[r], c.x[r] * c.x[r]));
            const float t = __builtin_fmaf(point.x, c.x[r], __builtin_fmaf(point.y, c.y[r], __builtin_fmaf(point.z, c.z[r], square)));
            const bool perhaps = t < upper && !(t < point.w) && (FULL || tile_index[p] < c.limit[r]);
            if (__ballot(perhaps) != 0) {
                const bool within = perhaps && exact(r, p);
                column[r] |= within ? bit : 0u;
                const uint32_t more = __popcll(__ballot(within));
                rows += lane == p ? more : 0u;
            }
        }
    }
}

} // namespace vesin_hip

#endif
