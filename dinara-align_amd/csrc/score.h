// Shared device/host definitions of the substitution-table (Scoring) kernels, score.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dinara {

// Below every reachable score: the host refuses pairs whose scores could come within a quarter of the 32-bit
// range (reference scoring.mojo:216-238, ScoreReach), so the sentinel plus a few steps never wraps or reads real.
constexpr int SCORE_NEG = -(1 << 28);

// What one launch of score_wave computes.
enum ScoreMode : int {
    SCORE_GLOBAL = 0,  // the corner's score
    SCORE_LOCAL = 1,   // the best cell, floored at zero, and where it lies
    SCORE_REACH = 2,   // over both prefixes reversed from a local end: the first cell reaching a target
    SCORE_TRACE = 3,   // the corner's score and every cell's decision, for the walk
};

// A pair takes a whole wave, or SCORE_NARROW lanes of one that then sweeps four pairs. A lane holds C columns: of a
// whole wave 1 to 8 in strips of 64C, of SCORE_NARROW lanes 1 to 16, one strip.
constexpr int SCORE_MAX_C = 8;
constexpr int SCORE_STRIP_MAX = 64 * SCORE_MAX_C;
constexpr int SCORE_NARROW = 16;
constexpr int SCORE_NARROW_COLS = 16 * SCORE_NARROW;

// A reference of more letters than the ring holds is read through it: chunks of this many letters, this many of them.
constexpr int SCORE_RING_CHUNK = 256;
constexpr int SCORE_RING_CHUNKS = 4;
constexpr int SCORE_RING = SCORE_RING_CHUNK * SCORE_RING_CHUNKS;

// Columns a lane of a whole wave: a strip of at most SCORE_STRIP_MAX columns, the strips as even as C allows.
__host__ __device__ inline int score_columns(int lanes, int cols) {
    if (lanes == SCORE_NARROW) return (cols + lanes - 1) / lanes;
    const int strips = (cols + SCORE_STRIP_MAX - 1) / SCORE_STRIP_MAX;
    const int per_strip = (cols + strips - 1) / strips;
    return (per_strip + 63) / 64;
}

// Bytes of one letter's scores against a lane's C columns: whole words, then a byte, a half or a word for the rest.
__host__ __device__ constexpr int score_tail(int c) { return c % 4 == 3 ? 4 : c % 4; }
__host__ __device__ constexpr int score_lane_bytes(int c) { return c / 4 * 4 + score_tail(c); }

struct ScoreArgs {
    const uint8_t *codes;    // every sequence's letter codes (the alphabet's places)
    const int64_t *ref_at;   // per slot: where its reference's codes start
    const int64_t *qry_at;   // per slot: where its query's codes start
    const int32_t *view;     // per slot: reference begin, reference letters, query begin, query letters
    int reversed;            // the views read both sequences back to front from their ends
    const int32_t *list;     // the slots of this launch, `count` of them
    int count;
    int lanes;               // lanes a pair: 64 or SCORE_NARROW
    int ref_room;            // LDS bytes for a pair's reference letters: SCORE_RING, or all of them and 4 more
    const int8_t *table;     // table[a * 32 + b]: reference letter a against query letter b
    int letters;
    int open, extend;        // a gap's first letter, each later one (scores, zero or less)
    int shifted;             // scores are held less `extend` for every row and column (extensions cost nothing)
    int mode;
    int end_bits;            // SCORE_LOCAL: > 0 keys each column's best as score << end_bits | row (rows and scores
                             // fit the 32 bits), 0 compares and selects
    int32_t *score;          // per slot
    int32_t *end_row;        // SCORE_LOCAL: the best cell's row and column; SCORE_REACH: the found cell's
    int32_t *end_col;
    const int32_t *target;   // SCORE_REACH: per slot, the score to reach
    uint32_t *arena;         // SCORE_TRACE: decisions, a wave's at arena_at[its place in the launch], in words
    const int64_t *arena_at;
    uint64_t *walk_base;     // SCORE_TRACE: per slot, the address of its decisions
    int32_t *walk_columns;   // SCORE_TRACE: per slot, the columns a lane its wave took
    int32_t *carry;          // the last column of a strip, two ints a row, a wave's at carry_at[..], in ints
    const int64_t *carry_at;
    // The walk's CIGARs (SCORE_TRACE only)
    int eqx;
    char *op_scratch;        // per slot, the walk's moves 2 bits each
    const int64_t *op_base;
    char *cigars;
    unsigned long long *cigar_used;
    int64_t *cigar_offset;
    int32_t *cigar_length;
    int slots;
};

// What a wave of `rows` by `cols` keeps (the largest of its pairs'): decision words, carry ints, LDS bytes.
inline int64_t score_decisions(int lanes, int64_t rows, int64_t cols) {
    const int c = score_columns(lanes, (int)cols);
    const int64_t strips = (cols + lanes * c - 1) / (lanes * c);
    return strips * (rows + lanes - 1) * ((c + 7) / 8) * 64;
}
inline int64_t score_carry(int lanes, int64_t rows, int64_t cols) {
    return lanes * score_columns(lanes, (int)cols) < cols ? 2 * (rows + 1) : 0;
}
inline size_t score_lds(int letters, int lanes, int cols, int ref_room) {
    return (size_t)letters * 64 * score_lane_bytes(score_columns(lanes, cols)) + (size_t)(64 / lanes) * ref_room;
}

// Host-side entry points of score.hip. `lds` is the bytes a block stages: the profile, then the references' letters.
void launch_score(const ScoreArgs &a, size_t lds, hipStream_t stream);
void launch_score_walk(const ScoreArgs &a, hipStream_t stream);

}  // namespace dinara
