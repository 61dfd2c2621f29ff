// The strip sweep (strip.hip): bands too wide for a group of sixteen lanes, two-piece gaps, free ends, and whole
// matrices, each pair cut into strips of columns that run as a pipeline of waves, and walked back by a whole wave.
#pragma once

#include "common.h"

namespace dinara {

// A strip is one wave, each lane holding C columns (2, 4 or 8).
__host__ __device__ constexpr int strip_columns(int c) { return 64 * c; }
// The persistent sweep's workgroups (a wave each): strips beyond them are claimed as waves finish theirs.
constexpr int STRIP_GRID = 8192;
// A wave's wait for its left strip's boundary column gives up after this many polls instead of hanging: its pair stays
// unsettled, as do the strips right of it and those no wave is left to claim, and `expired` says so.
constexpr int STRIP_POLL_LIMIT = 1 << 22;

// One pair of a launch: the diagonals lo..hi it sweeps (query letters less reference letters) and its place in the
// launch's memory.
struct StripPair {
    int32_t slot;
    int32_t lo, hi;
    int32_t c;            // columns a lane
    int32_t strips;
    int32_t rows;         // the rows a strip's records have room for
    int64_t decision_at;  // its first decision byte
    int64_t carry_at;     // its first carry word
};

// Strip `strip` of a pair of `n` reference letters: the rows whose cells of the strip's columns hold the band.
__host__ __device__ inline int strip_first_row(const StripPair &p, int strip) {
    const int64_t row = (int64_t)strip * strip_columns(p.c) + 1 - p.hi;
    return row > 1 ? (int)row : 1;
}
__host__ __device__ inline int strip_last_row(const StripPair &p, int strip, int n) {
    const int64_t row = (int64_t)(strip + 1) * strip_columns(p.c) - p.lo;
    return row < n ? (int)row : n;
}
// The decision bytes a lane keeps a row: 4 bits a column under one gap piece, a byte under two.
__host__ __device__ constexpr int strip_record_bytes(int c, int pieces) { return pieces == 2 ? c : c / 2; }

struct StripArgs {
    SweepArgs s;               // the batch's tape, costs, certificate, results and CIGAR output
    const StripPair *pairs;
    const int2 *order;         // the launch's strips (pair, strip) as they are claimed (null: a strip a pair, in turn)
    int count, strips;         // the pairs and strips of the launch
    int whole;                 // the bands hold the whole matrices: every cost found settles its pair
    uint8_t *decisions;        // null: costs alone
    unsigned long long *carry; // per pair and strip, `rows` boundary records (two words with two pieces), zero: not
                               // yet written
    int *claim;                // the strips claimed so far (zero at launch)
    int polls;                 // a wait gives up after this many
    int *expired;              // the waits that gave up are added here (null: not counted)
    int *done;                 // free ends, per pair: the strips that have ended (zero at launch)
    unsigned long long *best;  // free ends, per pair: the least cost and its diagonal's rank (all ones at launch)
};

// Host-side entry points of strip.hip: the sweep of every strip, settling each pair or filing it for a wider band;
// then, for launches that keep decisions, the walk and CIGAR of each pair the launch settled, a wave a pair.
void launch_strip_sweep(const StripArgs &a, hipStream_t stream);
void launch_strip_walk(const StripArgs &a, hipStream_t stream);
// Lists the slots whose status is not settled (0) into `list`, their number into `count` (zero at launch).
void launch_collect_unsettled(const int32_t *status, int slots, int32_t *list, int32_t *count, hipStream_t stream);

}  // namespace dinara
