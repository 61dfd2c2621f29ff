// Shared device/host definitions of the MI355X alignment kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dinara {

// A cell no path inside the band reaches. Every real cost stays below REAL_LIMIT (the host refuses pairs
// whose dearest path could pass it), so INF plus a few moves never wraps and never reads as real.
constexpr int INF = 1 << 28;
constexpr int REAL_LIMIT = 1 << 26;

// Gap-affine costs in the sweep's terms (reference lanes.mojo:187-259, modes.mojo:35-195): a deletion, a
// reference letter alone, of k letters costs del_open + k * del_ext; an insertion ins_open + k * ins_ext.
struct CostParams {
    int mismatch;
    int del_open, del_ext, ins_open, ins_ext;
    int del_first, ins_first;  // a gap's first letter: opening plus extension
    // Two-piece costs (reference lanes.mojo:187-345): a gap costs the less of its two pieces; with one piece
    // (pieces == 1) the second's fields are unused.
    int pieces;
    int del_open2, del_ext2, ins_open2, ins_ext2;
    int del_first2, ins_first2;
};

// Zero words after the tape's last group, 64 a word index across the transposed groups. The unit-cost sweeps' letter
// cursors (edit.hip) read ahead with no bounds check, at most two word indices past their group's last: a cursor loads
// no word more than two past the one that holds its last letter; a query's last letter is m - 1, and a band starts no
// lower than diagonal -n - 1, so its bottom row's letters end at n + m, which the group's query words, lying behind its
// reference words, hold but for that same margin.
constexpr int TAPE_PADDING_WORDS = 4 * 64;

// Which pairs a launch takes and where their letters lie. The tape holds every sequence 2 or 8 bits a
// letter, 16 or 4 to a 32-bit word, transposed by groups of 64 slots: slot s (the s-th pair in length
// order) has word w of its reference at tape[group_base[s / 64] + w * 64 + s % 64], its query words after
// group_ref_words[s / 64] reference words.
struct Tape {
    const uint32_t *words;
    const int64_t *group_base;
    const int32_t *group_ref_words;
    const int32_t *rows;  // reference letters per slot
    const int32_t *cols;  // query letters per slot
    int bits;
};

// The sweep classes: four sixteen-lane-group bands (32, 64, 128, 256 diagonals, group.hip); wave-per-pair bands of
// 64Q (Q = 1..32, sweep.hip) for every pair under a user band; and strip bands (strip.hip), 512 to 16384 diagonals by
// width, which one launch a round takes together.
constexpr int CLASS_GROUP32 = 0;
constexpr int CLASS_GROUP64 = 1;
constexpr int CLASS_GROUP256 = 3;
constexpr int CLASS_WAVE_FIRST = 4;  // Q = 1, 2, 4, 8, 16, 32 for classes 4..9
constexpr int CLASS_WAVE_LAST = 9;
constexpr int CLASS_STRIP_FIRST = 10;
constexpr int STRIP_CLASSES = 12;
constexpr int CLASSES = CLASS_STRIP_FIRST + STRIP_CLASSES;
constexpr int CLASS_TOO_WIDE = -1;

// The diagonals a class's band holds (a strip class's at most: 512, 1024, 1536, 2048, 3072, 4096 .. 8192 in steps of
// 1024, 12288, 16384).
__host__ __device__ constexpr int band_width(int cls) {
    return cls <= CLASS_GROUP256      ? 32 << cls
           : cls <= CLASS_WAVE_LAST   ? 64 << (cls - CLASS_WAVE_FIRST)
           : cls < CLASS_STRIP_FIRST + 4 ? 512 * (cls - CLASS_STRIP_FIRST + 1)
           : cls < CLASS_STRIP_FIRST + 10 ? 1024 * (cls - CLASS_STRIP_FIRST - 1)
                                          : 4096 * (cls - CLASS_STRIP_FIRST - 7);
}
__host__ __device__ constexpr bool band_is_wave(int cls) { return cls >= CLASS_WAVE_FIRST && cls <= CLASS_WAVE_LAST; }
__host__ __device__ constexpr bool band_is_strip(int cls) { return cls >= CLASS_STRIP_FIRST; }

// Which pairs take which bands, in letters (both sequences; 0 where no pair takes them): group bands of up to 64
// diagonals up to `group_narrow`, of 128 up to `group128_letters`, of 256 up to `group_letters`; the wave band of 64
// diagonals up to `wave_letters` and that of 128 up to `wave128_letters`; strips up to `strip_letters` and bands
// `strip_widest` wide.
struct BandLimits {
    int group_narrow, group128_letters, group_letters, wave_letters, wave128_letters, strip_letters, strip_widest;
};

__host__ __device__ inline int group_limit(const BandLimits &limits, int cls) {
    return cls <= CLASS_GROUP64 ? limits.group_narrow : cls < CLASS_GROUP256 ? limits.group128_letters : limits.group_letters;
}

// The class of band a pair of `letters` letters needing `need` diagonals takes: the narrowest that holds them. A group
// band is placed on an even diagonal, so it holds one diagonal fewer than its width. Pairs under a user band take the
// wave bands, which bar diagonals outside it.
__host__ __device__ inline int band_class(int need, int64_t letters, bool user_band, const BandLimits &limits) {
    if (user_band) {
        for (int cls = CLASS_WAVE_FIRST; cls <= CLASS_WAVE_LAST; ++cls)
            if (need <= band_width(cls)) return cls;
        return CLASS_TOO_WIDE;
    }
    for (int cls = CLASS_WAVE_FIRST; cls <= CLASS_WAVE_FIRST + 1; ++cls)
        if (letters <= (cls == CLASS_WAVE_FIRST ? limits.wave_letters : limits.wave128_letters) && need <= band_width(cls))
            return cls;
    for (int cls = CLASS_GROUP32; cls <= CLASS_GROUP256; ++cls)
        if (need < band_width(cls) && letters <= group_limit(limits, cls)) return cls;
    if (letters <= limits.strip_letters)
        for (int cls = CLASS_STRIP_FIRST; cls < CLASSES; ++cls)
            if (need <= band_width(cls) && band_width(cls) <= limits.strip_widest) return cls;
    return CLASS_TOO_WIDE;
}

// Everything a sweep launch reads and writes.
struct SweepArgs {
    Tape tape;
    const int32_t *list;  // slots to sweep, `count` of them
    int count;
    int cls;              // the launch's band class
    int slots;            // slots in the batch
    int32_t *want_low;    // per slot: the lane diagonals (query less reference) the band must hold
    int32_t *want_high;
    CostParams costs;
    int strict;           // 1 for alignments: no path off the band may cost as little
    int64_t cap;          // the cost cap, or a value past every cost
    int user_band;        // 1 when diagonals outside [user_low, user_high] (lane terms) are barred
    int doubling;         // 1: an unproven pair's next band is its band twice as wide, not the band its cost proves
    int user_low, user_high;
    int eqx;
    int forward_cigar;    // 1 when the tape holds both sequences reversed (Ties.LEFT): moves come in order
    int record;
    int lds_limit;        // letters one wave kernel's LDS holds
    // results per slot
    int32_t *cost;
    int32_t *status;      // 0 settled, 1 filed for a wider band, 2 wider than any band class
    int32_t *walk_low;    // the settled band's lowest diagonal and its class, for the walk
    int32_t *walk_class;
    // decisions: a group band's 4 bits a cell, a word for each diagonal pair every 8 anti-diagonals; a wave band's
    // a byte a cell, W bytes a row
    uint8_t *arena;          // this launch's decisions, `arena_stride` bytes a listed pair
    int64_t arena_stride;
    uint64_t *walk_flags;    // per slot: the address of its settled band's decisions
    int group_letters;       // LDS bytes a pair takes in a group launch (four pairs a block)
    int group16_top;         // > 0: group launches of two slots a lane and more hold their steady cells as 16-bit
                             // halves, `group16_top` the unreachable value (letters then take 2 bytes each in LDS)
    BandLimits limits;       // which pairs take which bands
    // CIGARs: each slot's scratch run of 2(n+m)+2 bytes from cigar_scratch_base, compacted into `cigars` at an
    // offset taken from `cigar_used`
    char *cigar_scratch;
    const int64_t *cigar_scratch_base;
    char *cigars;
    unsigned long long *cigar_used;
    int64_t *cigar_offset;
    int32_t *cigar_length;
    // unproven slots, filed by the class of the band that will prove them
    int32_t *retry_lists;  // CLASSES lists of `retry_capacity` slots each
    int32_t *retry_counts;
    int retry_capacity;
    int4 *strip_retries;   // the slots filed for strip bands (counted at CLASS_STRIP_FIRST): slot, low, high, 0
    // Free ends (strip sweeps only). Each slot sweeps a view of its pair: view_rows reference letters from
    // view_ref_at and view_cols query letters from view_qry_at, read back to front when `view_reversed`; free[4 s ..
    // 4 s + 3] the letters it may leave out for nothing at the start and end of the view's reference, then at those
    // of its query. A settled slot's end cell (the least cost; ties to the highest diagonal, or the lowest with
    // `lowest_end`) goes to end_row / end_col.
    int free_ends;
    int view_reversed;
    int lowest_end;
    const int32_t *view_rows, *view_cols, *view_ref_at, *view_qry_at;
    const int32_t *free;
    int32_t *end_row, *end_col;
};

// Host-side entry points of sweep.hip.
int class_width(int cls);
bool class_is_wave(int cls);
void launch_sweep(const SweepArgs &a, size_t lds, hipStream_t stream);
void launch_walk(const SweepArgs &a, hipStream_t stream);
void launch_group(int s, const SweepArgs &a, size_t lds, hipStream_t stream);

}  // namespace dinara
