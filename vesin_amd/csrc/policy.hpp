// Host-side decisions of the driver that depend on a list's history, kept apart from the HIP code so that they can
// be compiled and tested on a machine without a GPU.
#ifndef VESIN_HIP_POLICY_HPP
#define VESIN_HIP_POLICY_HPP

#include <algorithm>
#include <cstddef>

namespace vesin_hip {

/// What a call was asked for besides the box: a remembered box is only a good guess for the same question again.
struct BoxKey {
    size_t n_points;
    double cutoff;
    int algorithm;
    bool full;
    bool sorted;

    bool operator==(const BoxKey& other) const {
        return n_points == other.n_points && cutoff == other.cutoff && algorithm == other.algorithm &&
               full == other.full && sorted == other.sorted;
    }
};

constexpr int BOX_REST = 32;       // calls without a guess after the first wrong one
constexpr int BOX_REST_MAX = 4096; // and after many wrong ones in a row

/// The grid is picked on the host from the box, which lives on the device: reading it costs a round trip before
/// anything else can be launched. A call may instead start from the box of the call before and check the guess at
/// its last synchronisation; a wrong guess costs a whole search. This is the bookkeeping of when to guess:
///  * only a call that asks what the call that stored the box asked (same number of points, cutoff, algorithm and
///    kind of list): another system is likely to bring another box, and a box that is much too small for the points
///    puts them all into a few cells;
///  * after a wrong guess the list does not guess for `BOX_REST` calls, and every further wrong guess in a row
///    doubles that time (up to BOX_REST_MAX), so that a trajectory whose box changes with every step stops paying;
///    a right guess brings the time back to BOX_REST.
struct BoxGuess {
    bool have_box = false; // a box is remembered (set by the call that read one from the device)
    BoxKey key = {0, 0.0, 0, false, false};
    int rest = 0;
    int next_rest = BOX_REST;

    /// Once per call, before anything else: does this call start from the remembered box?
    bool begin(const BoxKey& now) {
        const bool guess = have_box && rest == 0 && now.n_points > 0 && key == now;
        if (rest > 0) {
            rest -= 1;
        }
        return guess;
    }

    void was_right() {
        next_rest = BOX_REST;
    }

    void was_wrong() {
        rest = next_rest;
        next_rest = next_rest >= BOX_REST_MAX / 2 ? BOX_REST_MAX : 2 * next_rest;
    }

    /// The call read its box from the device and remembered it.
    void stored(const BoxKey& now) {
        key = now;
    }
};

constexpr int WAIT_REST = 64;        // calls that leave a launch with waiting workgroups alone after it gave up
constexpr int WAIT_REST_MAX = 4096;  // and after it gave up many times in a row

/// Some launches make workgroups wait for each other (the chain that places the rows of the single-pass search in
/// work-item order, the meeting of a small system's one launch). That only advances while the workgroups that are
/// waited for get to run, which holds on a GPU the launch has to itself and may not on one it shares with other
/// streams or processes. Every such wait is bounded, and a launch whose waves gave up is followed by the passes that
/// need no waiting; this is the bookkeeping that keeps a list from paying for the give-up on every call: after one,
/// the list leaves that launch alone for WAIT_REST calls, and every further give-up in a row doubles that, up to
/// WAIT_REST_MAX; a launch that went through brings the time back to WAIT_REST.
struct WaitRest {
    int rest = 0;
    int next_rest = WAIT_REST;

    /// Once per call that could use the launch: true while the list stays away from it.
    bool resting() {
        if (rest > 0) {
            rest -= 1;
            return true;
        }
        return false;
    }

    void gave_up() {
        rest = next_rest;
        next_rest = next_rest >= WAIT_REST_MAX / 2 ? WAIT_REST_MAX : 2 * next_rest;
    }

    void went_through() {
        next_rest = WAIT_REST;
    }
};

/// options.skin > 0: kept candidates pay when calls that only filter them outnumber the calls that compute them
/// again, which cost a failed filter and a search at cutoff + skin (two to three direct searches). A skin too thin
/// for how far the points move between calls turns that around, and in a batch, where one system past its limit
/// costs all systems their candidates, so does a large number of systems: candidates that serve fewer than
/// CANDIDATES_SHORT_LIVED filtering calls are short-lived, and after CANDIDATES_STRIKES such sets in a row the list
/// searches directly, keeping nothing, for CANDIDATES_REST calls before it tries candidates again. The rows are the
/// same either way.
constexpr int CANDIDATES_SHORT_LIVED = 4;
constexpr int CANDIDATES_STRIKES = 3;
constexpr int CANDIDATES_REST = 64;

struct CandidateLifetime {
    int filtered = 0; // calls that the current candidates served
    int strikes = 0;  // short-lived sets in a row
    int rest = 0;     // direct calls left before candidates are tried again

    void served() {
        filtered += 1;
    }

    /// The check found the candidates outdated. True: no new ones for a while.
    bool outdated() {
        strikes = filtered < CANDIDATES_SHORT_LIVED ? strikes + 1 : 0;
        filtered = 0;
        if (strikes >= CANDIDATES_STRIKES) {
            strikes = 0;
            rest = CANDIDATES_REST;
            return true;
        }
        return false;
    }

    /// Once per call without usable candidates: true while the list stays with the direct search.
    bool resting() {
        if (rest > 0) {
            rest -= 1;
            return true;
        }
        return false;
    }

    void reset() {
        filtered = 0;
        strikes = 0;
        rest = 0;
    }
};

// ---------------------------------------------------------------------------------------------------------------
// The search that writes a sorted list in order (ordered.cuh): how its work is cut into waves. Every choice gives
// the same list; the figures are what the passes were measured at on one MI355X (256 compute units, 1024 SIMDs).

constexpr unsigned int ORDERED_TILE_POINTS = 32; // the points a tile holds at most (TILE_POINTS of the kernels)

/// Points of a tile that one wave of the counting and the writing pass takes (a power of two, at most 32).
///
/// Large systems: a whole tile, and the candidates of every tile are put in order once by a launch of its own.
/// Systems of fewer than 2048 occupied cells (up to 3072 at 12 points per cell or fewer) are latency, not throughput:
/// either pass lasts as long as its slowest wave, which grows with the points the wave writes the rows of. Shares of
/// 8 points, of 4 where 8 would leave fewer than about 1300 waves with any points at all (per call, cutoff 5, full
/// lists, shares of 32 / 16 / 8 / 4 / 2 points: 10,000 atoms at 0.05 per cubic A 116 / 100 / 93 / 100 / 127 us, at
/// 0.1 137 / 125 / 101 / 108 / 115 us; 4,000 atoms 101 / 85 / 76 / 74 / 86 and 125 / 122 / 94 / 82 / 81 us). Shares
/// that most tiles have no points for cost next to nothing in time, their waves leave at once, but each has room for
/// its candidates' records: a caller with a fixed amount of work memory (`coarse`) keeps the rule for the smallest
/// systems only, which halves the share until every possible share of every tile slot makes 2048 waves.
inline unsigned int ordered_share(size_t n_points, size_t n_cells, size_t tile_slots, bool coarse) {
    unsigned int share = ORDERED_TILE_POINTS;
    const size_t occupied = n_cells < n_points ? n_cells : n_points;
    const double filled = occupied < 1 ? 1.0 : static_cast<double>(occupied);
    double mean = static_cast<double>(n_points) / filled;
    if (mean > ORDERED_TILE_POINTS) {
        mean = ORDERED_TILE_POINTS;
    }
    if (!coarse && (filled < 2048.0 || (filled < 3072.0 && mean <= 12.0))) {
        const double shares_of_eight = mean <= 8.0 ? 1.0 : (mean <= 16.0 ? 2.0 : (mean <= 24.0 ? 3.0 : 4.0));
        share = filled * shares_of_eight < 1300.0 ? 4 : 8;
    }
    while (share > 1 && tile_slots * (ORDERED_TILE_POINTS / share) < 2048) {
        share /= 2;
    }
    return share;
}

/// Whether the in-order search may take the work memory it asks for. Its counting pass leaves a record per
/// candidate for the writing pass, in a block of fixed size per tile *slot* (12 KB, room for 1024 candidates), and the
/// number of slots follows the cells as well as the points: a dense system takes about 1 KB per point (1,000,000
/// atoms of diamond: 0.9 GB), a sparse one with a cell per point would take 12 KB per point (17,000,000 points: 212
/// GB). Beyond 2 GiB + 1.5 KB per point the sorted list is made by the search for crowded cells, whose
/// records take the room their candidates need (under the same rule), or by the search without records and the radix sort.
inline bool ordered_records_fit(size_t n_points, size_t record_bytes) {
    const double allowed = 2147483648.0 + 1536.0 * static_cast<double>(n_points);
    return static_cast<double>(record_bytes) <= allowed;
}

/// Room for what the search for crowded cells leaves between its passes, in units of 64: candidates of every cell (8 bytes
/// each), hit columns of every tile (4 bytes per candidate).
struct CrowdedRoom {
    size_t candidate_units = 0; // 0: not known, or none
    size_t column_units = 0;
};

inline bool crowded_room_fits(size_t n_points, const CrowdedRoom& room) {
    return room.candidate_units <= 0xFFFFFFF0ull && room.column_units <= 0xFFFFFFF0ull &&
           ordered_records_fit(n_points, 64 * (8 * room.candidate_units + 4 * room.column_units));
}

/// The room for a system whose candidates and columns were counted: an eighth more than that, so that the next frame finds
/// room too, or just that where the rule allows no more. None when not even that fits.
inline CrowdedRoom crowded_room_for(size_t n_points, const CrowdedRoom& counted) {
    const CrowdedRoom ample = {
        counted.candidate_units + counted.candidate_units / 8 + 64, counted.column_units + counted.column_units / 8 + 64
    };
    return crowded_room_fits(n_points, ample) ? ample : crowded_room_fits(n_points, counted) ? counted : CrowdedRoom{};
}

/// The room that the next call on as many points starts from: what this call had, and more where its system comes near
/// that, as long as the two together fit.
inline CrowdedRoom crowded_room_kept(size_t n_points, const CrowdedRoom& had, const CrowdedRoom& counted) {
    const CrowdedRoom wanted = crowded_room_for(n_points, counted);
    const CrowdedRoom both = {
        had.candidate_units > wanted.candidate_units ? had.candidate_units : wanted.candidate_units,
        had.column_units > wanted.column_units ? had.column_units : wanted.column_units
    };
    return crowded_room_fits(n_points, both) ? both : had;
}

/// Whether the in-order search for crowded cells (crowded.cuh) is the faster way to a sorted list than the radix sort. It
/// gives every tile workgroups of its own, whatever the tile holds; the radix sort's time follows the rows and has a floor
/// of 0.2 ms. Per call, radix sort -> that search, cutoff 5, liquids of 300,000 points with 2 / 3 / 4 / 6 / 8 points per cell:
/// full lists i j S d 793 -> 1118, 869 -> 920, 1007 -> 762, 1279 -> 622, 1587 -> 545 us, half lists i j S d D 676 -> 1242,
/// 707 -> 1032, 764 -> 859, 909 -> 710, 1101 -> 628 us; 20,000 points with 0.3 / 1 / 4: 203 -> 202, 218 -> 182, 215 -> 126 us.
inline bool crowded_search_pays(size_t n_points, size_t n_tiles) {
    return n_tiles <= 16384 || n_points >= 5 * n_tiles;
}

/// Whether the search gives every tile a workgroup (ordered_tile.cuh) in place of a wave or several (ordered.cuh), from the
/// number of tiles the call before had on the same points (0: not known, and a wave per tile).
///
/// Its kernels are the faster ones but for many tiles of few points, where most of a workgroup has nothing to do: the more
/// tiles, the better the waves of the other way fill the chip by themselves, and the kernels of lists with vectors leave room
/// for fewer workgroups (write_tile.cuh). Full and half lists cross at the same points per tile. The line follows where both
/// ways took the same for liquids of 3,000 to 1,000,000 points (cutoffs 3.5 and 5): without vectors 1.5 points per tile at
/// 9,000 tiles, 2.8 at 14,400, 3.5 at 18,700, 5 from 59,000 on; with vectors 1.5 at 8,000, 2.4 at 10,600, 3.5 at 11,700, 5 to 6
/// from 16,400 on, 6.3 at 64,000. Calls, a wave per tile or share of one -> a workgroup per tile, us:
///  - below the line: full P S d D, 1.8 points in each of 16,400 tiles 162 -> 187, 2.8 of 14,400 164 -> 183, 4.1 of 72,800 588 ->
///    698; half P S d D, 2.0 of 15,400 153 -> 174, 6.3 of 63,900 657 -> 689; full P S d, 2.0 of 15,400 152 -> 163;
///  - above it: full P S d D, 5.7 of 10,600 193 -> 172; half P S d D, 7.6 of 39,300 524 -> 466; full P S d, 3.2 of 4,700 126 ->
///    105, 4.4 of 13,600 193 -> 172, 6.0 of 166,000 1725 -> 1518; 100,000 points, 26 per cell, half P S d D 297 -> 201;
///    1,000,000 atoms of diamond, full P S d 1615 -> 1287.
inline bool ordered_by_tiles(size_t n_points, size_t tiles_before, bool vectors) {
    const double points = static_cast<double>(n_points);
    const double tiles = static_cast<double>(tiles_before);
    const double wanted = !vectors         ? std::min(5.0, 1.5 + (tiles - 9000.0) / 4000.0)
                          : tiles > 40000.0 ? 6.5
                                            : std::min(6.0, 1.5 + (tiles - 8000.0) / 1300.0);
    return tiles_before > 0 && points >= std::max(1.5, wanted) * tiles;
}

/// How the writing passes with a workgroup per tile (write_tile.cuh) store their rows.
enum TileStores : int {
    STORE_CACHED,     // through the caches
    STORE_STREAMED,   // past them (non-temporal)
    STORE_BY_GRANULE, // past them, but for the granules of 16 rows that a run of consecutive rows starts or ends in
};

/// A run of consecutive rows starts and ends in the middle of 64-byte pieces that other workgroups write the rest of. Stored
/// past the caches, such a piece is written to memory twice, in parts, which costs several times what a whole one does;
/// stored through them it is put together, in the L2 or in the 256 MB behind it, if both parts come while it is there.
/// Whole pieces of lists larger than that are better off past the caches. Writing pass, past / through / by granule, us:
///  - up to 200 MB: 60,000 points, 12 per cell, full P S d 48 / 36 / 44, P S d D 68 / 48 / 55; 100,000 points, 15 per cell,
///    half P S d 57 / 44 / 56, 25 per cell, half P S 58 / 43 / 51; 30,000 points, 20 per cell, full P S d 37 / 30 / 33;
///  - beyond, with vectors: 100,000 points, 26 per cell, half P S d D 108 / 88 / 78; 300,000 points, 20 per cell, full P S D
///    377 / 428 / 309, P S d D 452 / 508 / 356;
///  - with distances: 150,000 points, 20 per cell, full P S d 146 / 151 / 106, 300,000 points 285 / 318 / 278, diamond of
///    110,592 atoms 107 / 101 / 84 and of 1,000,000 atoms 910 / 1020 / 810 (in random order 988 / 1255 / 1004); but 500,000
///    points, 12 per cell, half (25 rows per point) 252 / 242 / 295: with nearly every row in such a granule, sorting them
///    out is all that is left;
///  - pairs alone 122 / 175 / 150, pairs and shifts 217 / 246 / 224 (300,000 points): the second set of stores costs more
///    than it saves.
inline TileStores tile_stores(size_t n_points, size_t rows, bool shifts, bool distances, bool vectors) {
    const size_t row_bytes = 16 + (shifts ? 12 : 0) + (distances ? 8 : 0) + (vectors ? 24 : 0);
    if (rows <= (size_t(200) << 20) / row_bytes) {
        return STORE_CACHED;
    }
    return (vectors || distances) && rows / 40 >= n_points ? STORE_BY_GRANULE : STORE_STREAMED;
}

/// The same for crowded cells, whose tiles are written in the order of the cells: the two runs that share a granule are most
/// often far apart in time, so the granules that wait for their second part, one per point, have to stay in the 256 MB
/// behind the L2 together with what else goes there. Without vectors sorting them out costs more than it saves. Calls on
/// clusters, past the caches / by granule, us: full P S d D, 50,000 points (20 M rows) 675 / 638, 100,000 (16 M) 589 / 559,
/// 300,000 (25 M) 843 / 872, 500,000 (58 M) 1349 / 1470, (82 M) 1782 / 1825; half 100,000 (11 M) 552 / 516, 500,000 (29 M) 1157 / 1260;
/// full P D, 300,000 (25 M) 802 / 838; P d, 500,000 points, writing pass 667 / 803.
inline TileStores crowded_stores(size_t n_points, size_t rows, bool shifts, bool distances, bool vectors) {
    const TileStores stores = tile_stores(n_points, rows, shifts, distances, vectors);
    const size_t granule_bytes = 16 * (16 + (shifts ? 12 : 0) + (distances ? 8 : 0) + 24);
    const bool stay = n_points <= (size_t(128) << 20) / granule_bytes;
    return stores == STORE_BY_GRANULE && !(vectors && stay) ? STORE_STREAMED : stores;
}

constexpr size_t BACKWARD_ROWS = 8192;    // of a workgroup at most
constexpr size_t BACKWARD_STEP = 512;     // and a multiple of this
constexpr size_t BACKWARD_RESIDENT = 512; // workgroups at a time: two on each of 256 compute units

/// Rows that one workgroup of the gradient's kernel (backward.cuh) takes. Many rows let more additions meet in its table
/// (1,000,000 atoms of diamond, 89 M rows, gradient of the distances: 1190 / 1098 / 1064 us with 2048 / 4096 / 8192 rows, 1101
/// with 16384). The rows are dealt out evenly over as few times BACKWARD_RESIDENT workgroups as that allows, but at least
/// two: a last round of a few workgroups takes as long as a full one. Powers of two, 512 to 1,023 workgroups up to 8.4 M rows
/// -> dealt out evenly, us: 0.7 M rows, half list, gradient of the distances and the box 46 -> 46; 2.7 M rows, full list,
/// distances 74 -> 66, vectors 75 -> 66; 4.5 M rows 113 -> 92 and 110 -> 90; 6.3 M rows 144 -> 122 and 138 -> 114, points in no
/// order 728 -> 688; 13.6 M rows 244 -> 231; 36 M rows 584 -> 580. (At least one round: half lists of 0.7 M rows 46 -> 38, but
/// points in no order 1.4 M rows 106 -> 124, where two rounds take 100.)
inline size_t backward_rows_per_block(size_t n_pairs) {
    const size_t most = BACKWARD_RESIDENT * BACKWARD_ROWS;
    const size_t rounds = std::max<size_t>(2, n_pairs / most + (n_pairs % most != 0));
    const size_t rows = (n_pairs - 1) / (BACKWARD_RESIDENT * rounds) + 1;
    return (rows + BACKWARD_STEP - 1) / BACKWARD_STEP * BACKWARD_STEP;
}

} // namespace vesin_hip

#endif
