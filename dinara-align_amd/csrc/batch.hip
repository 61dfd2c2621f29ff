// The C ABI's batch calls under `dinara_costs`: validation with the reference's result codes, packing into the
// device tape, the sweep launches class by class until every pair is proven, and results in the caller's
// order. Reference behaviour followed: c/dinara.mojo:111-190 (argument parsing and codes), :96-108 (per-pair
// refusals), :563-819 (batch results), lanes.mojo:1163-1252 (first band), api.mojo:1188-1213 (alignments).

#include <algorithm>
#include <chrono>
#include <functional>
#include <atomic>
#include <memory>
#include <new>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <numeric>
#include <optional>
#include <thread>
#include <vector>

#include "../../include/dinara.h"
#include "carved.h"
#include "common.h"
#include "device.h"
#include "edit.h"
#include "host.h"
#include "learned.h"
#include "strip.h"

using namespace dinara;

namespace {

constexpr int64_t UNBOUNDED = int64_t(1) << 60;
constexpr int64_t MAX_COST = int64_t(1) << 32;

// The costs a batch asked for, checked as the reference checks them (modes.mojo:84-143); `code` is nonzero
// when the batch fails whole.
struct ParsedCosts {
    int64_t code = 0;
    int64_t mismatch = 1, opening = 0, extension = 1, del_opening = 0, del_extension = 1;
    bool two_piece = false;
    // The second pieces when two_piece (reference modes.mojo:99-143): a side given none counts its one piece twice.
    int64_t opening2 = 0, extension2 = 1, del_opening2 = 0, del_extension2 = 1;
};

ParsedCosts parse_costs(const dinara_costs *c) {
    ParsedCosts p;
    if (!c) return p;  // unit costs
    auto invalid = [&]() {
        p.code = DINARA_INVALID_COSTS;
        return p;
    };
    if (c->mismatch <= 0 || c->extension <= 0 || c->opening < 0) return invalid();
    if (c->mismatch > MAX_COST || c->opening > MAX_COST || c->extension > MAX_COST) return invalid();
    p.mismatch = c->mismatch;
    p.opening = c->opening;
    p.extension = c->extension;
    p.del_opening = c->opening;
    p.del_extension = c->extension;
    if (c->opening2 >= 0) {
        if (c->extension2 <= 0) return invalid();
        if (c->opening2 > MAX_COST || c->extension2 > MAX_COST) return invalid();
        p.two_piece = true;
        p.opening2 = c->opening2;
        p.extension2 = c->extension2;
    }
    p.del_opening2 = p.opening2;
    p.del_extension2 = p.extension2;
    if (c->deletion_extension != 0) {
        if (c->deletion_extension <= 0 || c->deletion_opening < 0) return invalid();
        if (c->deletion_opening2 >= 0 && c->deletion_extension2 <= 0) return invalid();
        if (c->deletion_opening > MAX_COST || c->deletion_extension > MAX_COST) return invalid();
        if (c->deletion_opening2 > MAX_COST || c->deletion_extension2 > MAX_COST) return invalid();
        p.del_opening = c->deletion_opening;
        p.del_extension = c->deletion_extension;
        if (c->deletion_opening2 >= 0) {
            p.del_opening2 = c->deletion_opening2;
            p.del_extension2 = c->deletion_extension2;
            if (!p.two_piece) {  // insertions gain a second piece: their own once more
                p.opening2 = p.opening;
                p.extension2 = p.extension;
            }
            p.two_piece = true;
        } else {
            p.del_opening2 = p.del_opening;  // deletions lack one: their own once more
            p.del_extension2 = p.del_extension;
        }
    }
    return p;
}

// The mode: global is all this library serves under Costs. Invalid modes are refused as the reference refuses
// them (modes.mojo:261-386, c/dinara.mojo:130-151); valid ones it does not serve as DINARA_INVALID_MODE.
int64_t check_mode(const dinara_mode *m) {
    if (!m) return 0;
    if (m->kind == DINARA_EXTENSION) {
        if (m->match_score < 0 || m->match_score > MAX_COST) return DINARA_INVALID_COSTS;
        return DINARA_INVALID_MODE;
    }
    if (m->kind == DINARA_LOCAL) {
        if (m->match_score < 0 || m->match_score > MAX_COST) return DINARA_INVALID_COSTS;
        return DINARA_INVALID_MODE;
    }
    if (m->kind != DINARA_ENDS_FREE) return DINARA_INVALID_MODE;
    if (std::min(std::min(m->reference_start, m->reference_end), std::min(m->query_start, m->query_end)) < 0)
        return DINARA_INVALID_MODE;
    if (m->match_score < 0 || m->match_score > MAX_COST) return DINARA_INVALID_COSTS;
    // Free ends that minimize the costs are served; a match score (maximized) is not.
    if (m->match_score > 0) return DINARA_INVALID_MODE;
    return 0;
}

// Whether a valid mode frees any letters at an end (reference modes.mojo:261-386: ends_free and its presets).
bool free_mode(const dinara_mode *m) {
    return m && (m->reference_start | m->reference_end | m->query_start | m->query_end) != 0;
}

struct Options {
    int64_t band_low = -UNBOUNDED, band_high = UNBOUNDED;  // library terms: reference less query letters
    int64_t max_cost = -1;
    bool eqx = true;
    bool right_ties = false;
};

Options parse_options(const dinara_options *o) {
    Options p;
    if (!o) return p;
    p.band_low = std::min(std::max(o->band_low, -UNBOUNDED), UNBOUNDED);
    p.band_high = std::min(std::max(o->band_high, -UNBOUNDED), UNBOUNDED);
    p.max_cost = o->max_cost;
    p.eqx = o->eqx != 0;
    p.right_ties = o->right_ties != 0;
    return p;
}

// Zero for a pair the library takes, else why not (reference c/dinara.mojo:96-108).
int64_t pair_code(const char *ref, int64_t n, const char *qry, int64_t m) {
    if (n < 0 || m < 0) return DINARA_INVALID_LENGTH;
    auto plain = [](const char *s, int64_t len) {
        const unsigned char *u = reinterpret_cast<const unsigned char *>(s);
        unsigned refused = 0;  // no early exit: the loop vectorizes
        for (int64_t i = 0; i < len; ++i) refused |= u[i] >= 0xFE;
        return refused == 0;
    };
    if ((n > 0 && !plain(ref, n)) || (m > 0 && !plain(qry, m))) return DINARA_UNSUPPORTED_SYMBOLS;
    return 0;
}

}  // namespace

// ------------------------------------------------------------------ the batch

// A strip round's parts, one launch each: consecutive pairs of its plan, and the memory the largest takes.
struct StripPart {
    size_t pair, pairs, strip, strips;
    size_t decision_bytes, carry_words;
};
struct StripParts {
    std::vector<StripPart> parts;
    size_t pairs = 0, decision_bytes = 0, carry_words = 0;
    int64_t class_pairs[CLASSES] = {};  // by the class of its band's width
};

struct dinara_batch {
    int gpu = 0;
    int64_t kind = DINARA_BATCH_DISTANCES;
    int64_t pairs = 0;
    int64_t threads = 0;
    Options options;
    ParsedCosts parsed;
    CostParams costs{};
    bool user_band = false;
    int user_low = 0, user_high = 0;
    int initial_width = 32;
    std::vector<int64_t> code;            // per pair: 0 on the device, else its own result code
    std::vector<int64_t> reference_length, query_length;
    std::vector<uint8_t> plain;           // per pair: 1 when its letters are A, C, G and T alone
    std::vector<int32_t> slot_pair;       // slot -> pair
    std::vector<int32_t> rows, cols;      // per slot
    std::vector<int32_t> first_low, first_high;
    std::vector<int32_t> first_lists[CLASSES];
    std::vector<int64_t> scratch_base;
    int bits = 2;
    bool reversed = false;                // the tape holds both sequences back to front (Ties.LEFT)
    bool doubling = false;                // retries double the band rather than take the band the cost proves
    size_t lds_limit = 0;
    DeviceContext *ctx = nullptr;
    int max_letters = 0;                  // the most letters of a pair, both sequences
    int32_t max_rows = 0;
    int group16_top = 0;                  // > 0: packed 16-bit group cells, this the unreachable value
    BandLimits limits{};                  // which pairs take which bands
    int64_t dearest = 1;                  // the dearest single step: a substitution or a gap's first letter
    // Free ends (wave sweeps): the letters each end of each sequence may leave out (reference start, end, query
    // start, end), the phase a run is in (1 the forward phase finding cost and end, 2 the anchored phase keeping
    // decisions), and per slot its views, free letters and first bands of each phase.
    bool free_ends = false;
    int64_t ends[4] = {0, 0, 0, 0};
    int phase = 0;
    std::vector<int32_t> a_rows, a_cols, a_at, a_free, a_first_low, a_first_high, a_first_all;
    std::vector<int64_t> a_first_offset;
    std::vector<int32_t> a_status_h, a_cost_h, a_end_row_h, a_end_col_h, b_end_row_h, b_end_col_h;
    std::vector<int32_t> b_rows_h, b_cols_h;
    std::vector<DeviceBuffer *> arenas;   // one per launch of a run, kept from run to run
    std::vector<int64_t> first_offset;    // where each class's first list starts in first_lists_d
    // device memory
    DeviceBuffer tape, group_base, group_ref_words, rows_d, cols_d, want_low, want_high, first_low_d,
        first_high_d, cost, status, walk_low, walk_class, cigar_scratch, cigar_scratch_base, cigars, cigar_used,
        cigar_offset, cigar_length, retry_lists, retry_counts, first_lists_d, walk_flags, view_rows_d, view_cols_d,
        view_ref_at_d, view_qry_at_d, free_d, end_row_d, end_col_d;
    Region region;  // what most of the buffers lie in
    ~dinara_batch() {
        for (DeviceBuffer *buffer : arenas) delete buffer;
        if (edit_graph) (void)hipGraphExecDestroy(edit_graph);
        if (region.base) give_back(ctx, region);
    }
    // the last run's results, by slot
    std::vector<int32_t> cost_h, status_h, cigar_length_h;
    std::vector<int64_t> cigar_offset_h;
    std::vector<char> cigars_h;
    bool ran = false;
    // statistics of the last run
    double run_ms = 0, sweep_ms = 0, walk_ms = 0, launches = 0, first_proven = 0;
    double class_ms[CLASSES] = {}, class_launches[CLASSES] = {}, class_pairs[CLASSES] = {};

    // The unit-cost path (edit.hip): unit costs times `unit_scale` and no user band.
    bool unit = false;
    int unit_scale = 1;
    bool use_graph = true;                // replay the run's launches as one captured hipGraph
    bool persistent = true;               // pair groups refill from their queue; else one pair a group
    bool keep_first = false;              // alignments: every sweep keeps its decisions (one pass when proven)
    bool side_by_side_bins = true;        // every one-word bin in one launch, the wider ones beside it
    bool one_stream = false;              // no side streams: the wider bins' launches follow on the main stream
    bool timed = true;                    // launches made one by one record an event pair each
    int grid_per_cu = 8;                  // persistent workgroups a compute unit
    int start_bin[EDIT_LENGTH_CLASSES] = {};  // the least first bin, by the pair's longer side
    uint32_t first_bins = EDIT_ALL_BINS;  // the bins a first band may take (bit b for bin b): the first pass's edges
    std::vector<int32_t> edit_first_low;  // per slot: its first band's lowest diagonal
    std::vector<int32_t> edit_first_bin;
    int64_t first_count[EDIT_BINS] = {};  // pairs each bin's first queue holds
    int64_t retry_reach[EDIT_BINS] = {};  // pairs a bin's retry queue may get: first bin narrower, widest no narrower
    int64_t trace_reach[EDIT_BINS] = {};  // pairs a bin's tracing sweep may meet
    DeviceBuffer features_d, predictions_d;  // learned seeding on the device
    int seeded_start[EDIT_LENGTH_CLASSES] = {-1};  // the start bins the device seeding's launch shape was made for
    DeviceBuffer edit_band_low, edit_first_low_d, edit_lists, edit_retry_lists, edit_retry_counts, edit_later_lists,
        edit_later_counts, edit_counts, edit_first_lists, edit_first_counts, trace_lists,
        trace_counts, trace_offset, walk_ready, walk_moves, walk_early, deferred, deferred_count, deferred_held,
        arena_used, edit_stats, edit_work;
    size_t arena_capacity = 0;            // the bytes of the context's arena this batch's runs use
    const void *arena_ptr = nullptr;      // where that arena was when the captured graph was made
    size_t arena_ask = 0, arena_bound = 0;  // the bytes it asks for and the most it may use (0: not worked out yet)
    hipGraphExec_t edit_graph = nullptr;
    double edit_ms[EDIT_BINS] = {}, trace_ms[EDIT_BINS] = {}, edit_sweeps[EDIT_BINS] = {},
           trace_sweeps[EDIT_BINS] = {}, graph_used = 0, trace_passes = 0, walked_first = 0;
    double sweep_work[EDIT_BINS] = {}, trace_work[EDIT_BINS] = {};  // word-columns swept by each bin
    bool stats_pending = false;  // the unit path's device counters of the last run, read when first asked for
    int64_t stats_slots = 0;
    // The whole-matrix path (strip.hip) for pairs the band sweeps leave unsettled: whether any pair is long enough
    // to need it (-1 not worked out yet), and the last run's count and time.
    int may_need_full = -1;
    bool expired = false;  // a strip's wait gave up in the last run: it left pairs to the whole-matrix path
    bool whole = false;  // every pair takes the whole-matrix path, no band sweep (for checking and comparison)
    double full_pairs = 0, full_ms = 0;
    DeviceBuffer full_list, full_count;
    // The strip launches' plan (pairs, then the order their strips are claimed in) and memory, and the slots filed for
    // strip bands (two sets taking turns, as the retry lists).
    DeviceBuffer strip_plan, strip_counts, strip_best, strip_carry, strip_decisions, strip_retries;
    // The first round's plan, on the device as long as the first bands stand (seeding moves them).
    DeviceBuffer first_strip_plan;
    StripParts first_strips;
    bool first_strips_planned = false;
};

namespace {

int64_t unit_lists(dinara_batch *b);
int64_t unit_buffers(dinara_batch *b, const std::vector<int32_t> &lists, const std::vector<int32_t> &counts,
                     size_t cap);

// Letters' room a group pair stages besides its own (sweep_group): 132 before, 9 between and 131 past; and its LDS bytes
// (twice as many in packed cells) where the launch's longest pair has `letters`.
constexpr int GROUP_ROOM = 272;
constexpr int64_t LDS_BYTES = 160 << 10;  // a compute unit's
int group_region(int64_t letters) { return (int)((letters + GROUP_ROOM + 3) & ~int64_t(3)); }

// Which pairs take which bands (prepare).
//
// A group launch is four pairs a wave, each a chain over its anti-diagonals: it takes as long as its longest pair, at
// any number of pairs up to a wave on each SIMD. A strip round takes as long as its strips' cells, as long as a group
// chain of as many letters as so many pairs' on average (CIGARs, whose strips write more decisions, have their own). So
// of the pairs past GROUP_LETTERS letters the longest go to the strips, down to the length that makes the two least
// together. Groups against strips, ms: 1,000 pairs of 1.2 kbp at 5% 0.79 and 0.81 (CIGARs 2.8 and 2.8), of 2 kbp 1.5 and
// 1.2 (5.8 and 3.5); 500 of 2.5 kbp at 1% 1.2 and 1.2 (4.2 and 4.0), 2,000 of 5 kbp 4.9 and 3.1 (13.0 and 9.1), 4,096 of
// 2.5 kbp 2.0 and 1.9 (6.8 and 7.9), 20,000 of 2.5 kbp 3.1 and 5.5 (12.5 and 21.3).
// In 128 diagonals the groups' cells are the fewer: 1,000 CIGARs of 1.8 kbp at 1% 3.1 and 3.5.
constexpr int64_t GROUP_LETTERS = 3072, GROUP128_LETTERS = 4608, GROUP_PAIRS_COSTS = 4096, GROUP_PAIRS_CIGARS = 3072;
// The first band is a narrow group band, a short chain that proves a pair of few errors; a pair's first strips are wide
// (first_strip_band), and prove more. What CIGARs take either way, in ns a letter of the longest pair (a group's sweep
// and its walks, a lane a pair; a strip round's sweep and its walks, a wave a pair) and of all pairs in strips: 64 pairs
// of 2.5 kbp at 1% 3.3 ms as groups and 1.5 as strips; at 0.1% 300 of 1.8 kbp 2.0 and 1.6, 1,000 of 2.2 kbp 2.8 and 5.1.
constexpr double GROUP_SWEEP_NS = 86, GROUP_WALK_NS = 350, STRIP_CHAIN_NS = 250, STRIP_WORK_NS = 0.8;

// The narrowest wave band, a row a step of a pair's own wave, against one strip of the whole matrix and its 63 steps of
// lanes coming in and going out: the pairs whose strips would take longer than the longest pair's rows. Two pieces, wave
// against strips, ms: 20,000 pairs of 150 bp 0.67 and 1.12, 3,000 of 600 0.97 and 1.10, 5,000 of 1,000 1.7 and 2.6, 1,000
// of 1,500 at 0.5% 1.6 and 1.3. The next wider one takes the same pairs' retries (5,000 CIGARs of 1,000 4.9 -> 4.5), under
// free ends, whose first bands are wide, short pairs alone: reads of 100 with a free reference end 0.69 and 1.03. CIGARs
// of these bands are walked a lane a pair, a chain of its own at the run's end: they pay where the strips they spare would
// take as long, from so many pairs on (1,000 two-piece CIGARs of 1.5 kbp, of which a few are short, 10.4 and 10.0).
constexpr int64_t WAVE_LETTERS = 512, WAVE_LETTERS_MOST = 8192, WAVE_PAIRS = 2560, WAVE128_LETTERS = 320,
                  WAVE_PAIRS_CIGARS = 450;

// The class of a slot's first band of `need` diagonals.
int first_class(const dinara_batch *b, int64_t s, int need) {
    return band_class(need, (int64_t)b->rows[s] + b->cols[s], b->user_band, b->limits);
}

// Builds the tape: pairs by length, longest first, 64 to a group, each group's words transposed.
int64_t prepare(dinara_batch *b, const char *const *refs, const char *const *qrys) {
    const int64_t pairs = b->pairs;
    std::vector<int32_t> order;
    order.reserve(pairs);
    for (int64_t i = 0; i < pairs; ++i)
        if (b->code[i] == 0) order.push_back((int32_t)i);
    longest_first(order, [&](int32_t p) { return (uint32_t)std::max(b->reference_length[p], b->query_length[p]); });
    const int64_t slots = (int64_t)order.size();
    b->slot_pair = order;
    b->first_offset.assign(CLASSES + 1, 0);
    if (slots == 0) return 0;  // every pair answered by its own code
    b->rows.resize(slots);
    b->cols.resize(slots);
    for (int64_t s = 0; s < slots; ++s) {
        b->rows[s] = (int32_t)b->reference_length[order[s]];
        b->cols[s] = (int32_t)b->query_length[order[s]];
    }
    // Two bits a letter when every pair holds at most four distinct bytes (each pair its own codes: only equality
    // counts), else a byte a letter.
    std::atomic<bool> wide{false};
    const bool all_plain = std::all_of(order.begin(), order.end(), [&](int32_t p) { return b->plain[p] != 0; });
    parallel_for(all_plain ? 0 : slots, b->threads, [&](int64_t lo, int64_t hi) {
        for (int64_t s = lo; s < hi; ++s) {
            const int32_t p = order[s];
            if (b->plain[p] || wide.load(std::memory_order_relaxed)) continue;
            bool present[256] = {false};
            int distinct = 0;
            auto scan = [&](const char *text, int64_t len) {
                const unsigned char *u = reinterpret_cast<const unsigned char *>(text);
                for (int64_t i = 0; i < len && distinct <= 4; ++i)
                    if (!present[u[i]]) {
                        present[u[i]] = true;
                        ++distinct;
                    }
            };
            scan(refs[p], b->reference_length[p]);
            scan(qrys[p], b->query_length[p]);
            if (distinct > 4) wide.store(true);
        }
    });
    b->bits = wide.load() ? 8 : 2;
    const int per = 32 / b->bits;
    const int64_t groups = (slots + 63) / 64;
    std::vector<int64_t> gbase(std::max<int64_t>(groups, 1));
    std::vector<int32_t> gref(std::max<int64_t>(groups, 1)), gqry(std::max<int64_t>(groups, 1));
    int64_t words = 0;
    for (int64_t g = 0; g < groups; ++g) {
        int32_t rw = 0, qw = 0;
        for (int64_t s = g * 64; s < std::min(slots, (g + 1) * 64); ++s) {
            rw = std::max<int32_t>(rw, (b->rows[s] + per - 1) / per);
            qw = std::max<int32_t>(qw, (b->cols[s] + per - 1) / per);
        }
        gbase[g] = words;
        gref[g] = rw;
        gqry[g] = qw;
        words += (int64_t)(rw + qw) * 64;
    }
    // Every word is written below (a pair's words past its letters are zero), so the tape needs no clearing but
    // its padding, where the unit-cost sweeps' unchecked letter reads past the last group land (TAPE_PADDING_WORDS).
    const int64_t padded = words + TAPE_PADDING_WORDS;
    std::unique_ptr<uint32_t[]> tape(new (std::nothrow) uint32_t[padded]);
    if (!tape) return DINARA_OUT_OF_MEMORY;
    std::fill(tape.get() + words, tape.get() + padded, 0u);
    // Ties.LEFT is the rule over both sequences reversed, so their tape is reversed (lanes.mojo:1523-1525).
    const bool reversed = b->kind == DINARA_BATCH_ALIGNMENTS && !b->options.right_ties && !b->free_ends;
    b->reversed = reversed;
    parallel_for(groups, b->threads, [&](int64_t lo, int64_t hi) {
        for (int64_t g = lo; g < hi; ++g) {
            const int64_t first = g * 64, last = std::min(slots, (g + 1) * 64);
            for (int64_t s = first; s < (g + 1) * 64; ++s) {
                uint32_t *ref_out = tape.get() + gbase[g] + (s & 63);
                uint32_t *qry_out = ref_out + (int64_t)gref[g] * 64;
                if (s >= last) {  // the group's empty slots
                    for (int32_t w = 0; w < gref[g]; ++w) ref_out[(int64_t)w * 64] = 0;
                    for (int32_t w = 0; w < gqry[g]; ++w) qry_out[(int64_t)w * 64] = 0;
                    continue;
                }
                const int32_t p = order[s];
                const int64_t n = b->reference_length[p], m = b->query_length[p];
                if (b->bits == 2 && b->plain[p]) {
                    // A, C, G and T are codes 0, 1, 2, 3 in every pair (the k-mer features read them so).
                    Dna::pack2(refs[p], n, reversed, ref_out, gref[g]);
                    Dna::pack2(qrys[p], m, reversed, qry_out, gqry[g]);
                    continue;
                }
                // Two-bit codes for a pair with other bytes: A, C, G and T keep 0, 1, 2, 3, any other byte the
                // least code its pair leaves free; or a byte a letter. Only equality counts to the sweeps.
                int16_t codes[256];
                for (int i = 0; i < 256; ++i) codes[i] = b->bits == 8 ? (int16_t)i : -1;
                if (b->bits == 2) {
                    bool used[4] = {false, false, false, false};
                    auto fixed = [](unsigned char byte) { return byte == 'A' ? 0 : byte == 'C' ? 1 : byte == 'G' ? 2 : byte == 'T' ? 3 : -1; };
                    auto note = [&](const char *text, int64_t len, bool fixed_pass) {
                        const unsigned char *u = reinterpret_cast<const unsigned char *>(text);
                        for (int64_t i = 0; i < len; ++i) {
                            if (codes[u[i]] >= 0) continue;
                            const int f = fixed(u[i]);
                            if (fixed_pass && f >= 0) {
                                codes[u[i]] = (int16_t)f;
                                used[f] = true;
                            } else if (!fixed_pass) {
                                int free_code = 0;
                                while (used[free_code]) ++free_code;
                                codes[u[i]] = (int16_t)free_code;
                                used[free_code] = true;
                            }
                        }
                    };
                    note(refs[p], n, true);
                    note(qrys[p], m, true);
                    note(refs[p], n, false);
                    note(qrys[p], m, false);
                }
                auto pack = [&](const char *text, int64_t len, uint32_t *out, int32_t words_here) {
                    const unsigned char *u = reinterpret_cast<const unsigned char *>(text);
                    for (int32_t w = 0; w < words_here; ++w) {
                        uint32_t word = 0;
                        for (int i = 0; i < per; ++i) {
                            const int64_t at = (int64_t)w * per + i;
                            if (at >= len) break;
                            const unsigned char byte = reversed ? u[len - 1 - at] : u[at];
                            word |= (uint32_t)codes[byte] << (b->bits * i);
                        }
                        out[(int64_t)w * 64] = word;
                    }
                };
                pack(refs[p], n, ref_out, gref[g]);
                pack(qrys[p], m, qry_out, gqry[g]);
            }
        }
    });
    b->max_rows = 0;
    b->max_letters = 0;
    for (int64_t s = 0; s < slots; ++s) {
        b->max_rows = std::max(b->max_rows, b->rows[s]);
        b->max_letters = std::max<int>(b->max_letters, b->rows[s] + b->cols[s]);
    }
    // A group pair's LDS region: both sequences, and room for reads up to half the widest group band (256) before the
    // reference and past the query (group.hip). The group sweep holds costs times 16 with a tag and runs up to half its
    // widest band past the corner: every value it makes stays under 2^30. It holds one gap piece and no free ends.
    int64_t letters_in_all = 0;
    for (int64_t s = 0; s < slots; ++s) letters_in_all += (int64_t)b->rows[s] + b->cols[s];
    const auto longest_up_to = [&](int64_t cap) {
        int longest = 0;
        for (int64_t s = 0; s < slots; ++s)
            if (b->rows[s] + b->cols[s] <= cap) longest = std::max(longest, b->rows[s] + b->cols[s]);
        return longest;
    };
    b->limits = BandLimits{};
    if (b->parsed.two_piece || b->free_ends) {
        const int64_t cap = std::min(std::max(WAVE_LETTERS, letters_in_all / WAVE_PAIRS), WAVE_LETTERS_MOST);
        const int longest = longest_up_to(std::min(cap, (int64_t)b->lds_limit));
        int64_t letters_there = 0;
        for (int64_t s = 0; s < slots; ++s)
            if (b->rows[s] + b->cols[s] <= longest) letters_there += b->rows[s] + b->cols[s];
        if (b->kind != DINARA_BATCH_ALIGNMENTS || letters_there >= WAVE_PAIRS_CIGARS * longest) b->limits.wave_letters = longest;
        b->limits.wave128_letters =
            b->free_ends ? (int)std::min<int64_t>(b->limits.wave_letters, WAVE128_LETTERS) : b->limits.wave_letters;
    } else {
        const int64_t staged = (int64_t)(b->lds_limit / 4) - GROUP_ROOM - 4;
        const bool cigars = b->kind == DINARA_BATCH_ALIGNMENTS;
        std::vector<int32_t> longs;  // letters, most first
        int32_t longest = 0;         // of the others
        int64_t past = 0, past_longest = 0;  // letters of the pairs no group launch stages
        for (int64_t s = 0; s < slots; ++s) {
            const int32_t letters = b->rows[s] + b->cols[s];
            if (letters <= GROUP_LETTERS) {
                longest = std::max(longest, letters);
            } else if (letters <= staged) {
                longs.push_back(letters);
            } else {
                past += letters;
                past_longest = std::max<int64_t>(past_longest, letters);
            }
        }
        std::sort(longs.begin(), longs.end(), std::greater<int32_t>());
        // Of each length that may be the longest in group bands (all, then ever fewer of the long pairs): the chain of the
        // wider bands and the strips beside them, and for CIGARs of the first round and its walks.
        int64_t cap = GROUP_LETTERS, first_cap = staged, in_strips = 0;
        double least = 0, least_first = 0;
        for (size_t i = 0; i <= longs.size(); ++i) {
            const int64_t chain = i < longs.size() ? longs[i] : longest;
            const double cost = (double)chain + (double)in_strips / (cigars ? GROUP_PAIRS_CIGARS : GROUP_PAIRS_COSTS);
            const int64_t strip_longest = past_longest > 0 ? past_longest : i > 0 ? longs[0] : 0;
            const double first = std::max(GROUP_SWEEP_NS * chain, STRIP_CHAIN_NS * strip_longest +
                                                                      STRIP_WORK_NS * (past + in_strips)) +
                                 GROUP_WALK_NS * chain;
            if (i == 0 || cost < least) {
                least = cost;
                cap = std::max(chain, GROUP_LETTERS);
            }
            if (i == 0 || first < least_first) {
                least_first = first;
                first_cap = i == 0 ? staged : std::max(chain, GROUP_LETTERS);
            }
            if (i < longs.size()) in_strips += longs[i];
        }
        const auto tags_fit = [&](int longest) {
            return ((int64_t)longest + 2 * 256 + 8) * b->dearest < REAL_LIMIT ? longest : 0;
        };
        if (!cigars) first_cap = staged;
        b->limits.group_letters = tags_fit(longest_up_to(std::min(first_cap, cap)));
        b->limits.group128_letters =
            std::max(b->limits.group_letters, tags_fit(longest_up_to(std::min(first_cap, GROUP128_LETTERS))));
        b->limits.group_narrow = std::max(b->limits.group128_letters, tags_fit(longest_up_to(first_cap)));
    }
    // The strips take bands of pairs up to 65,536 letters, free ends' up to 2,048 diagonals; longer pairs and wider
    // bands are swept whole after the run.
    b->limits.strip_letters = 65536;
    b->limits.strip_widest = b->free_ends ? 2048 : band_width(CLASSES - 1);
    // Packed 16-bit group cells (group.hip) for shifted costs (equal extensions e) whose mismatch is no dearer than
    // two extension letters: a tagged value then lies in [-16 e (n + m), 32 opening + 15]. A cell no path reaches starts
    // at `top` on the two anti-diagonals before (0, 0)'s and loses at most 32 e a diagonal step: on anti-diagonal t it
    // stays at or above `top` - 16 e (t + 2). So both fit 16 bits, apart, while 16 e (n + m + 2) + 32 opening + 15 stays
    // under `top` (less a margin); `top` leaves room for an opening's add, and the seed's 32 e fits with it.
    // DINARA_GROUP_CELLS32 set keeps 32-bit cells, for comparison.
    b->group16_top = 0;
    {
        const CostParams &k = b->costs;
        const int64_t e = k.del_ext, opening = std::max(k.del_open, k.ins_open);
        const int64_t top = (32767 - 16 * opening - 32) & ~int64_t(15);
        const int64_t longest = b->limits.group_letters;
        if (longest > 0 && !std::getenv("DINARA_GROUP_CELLS32") && k.pieces != 2 && k.del_ext == k.ins_ext &&
            e >= 0 && k.mismatch >= 0 && k.mismatch <= 2 * e && std::min(k.del_open, k.ins_open) >= 0 &&
            16 * e * (longest + 2) + 32 * opening + 15 < top - 64 && (size_t)8 * group_region(longest) <= b->lds_limit)
            b->group16_top = (int)top;
    }
    // The first band: the lanes' start and end diagonals and one either side (lanes.mojo:1207-1215), within the
    // user band; swept at no less than the initial width, centred.
    b->first_low.resize(slots);
    b->first_high.resize(slots);
    for (auto &l : b->first_lists) l.clear();
    if (b->free_ends) b->a_free.assign((size_t)slots * 4, 0);
    b->scratch_base.resize(slots + 1);
    int64_t scratch = 0, text = 0;
    for (int64_t s = 0; s < slots; ++s) {
        const int32_t n = b->rows[s], m = b->cols[s];
        const int32_t end = m - n;
        int32_t lo = std::min(0, end) - 1, hi = std::max(0, end) + 1;
        if (b->user_band) {
            lo = std::max(lo, b->user_low);
            hi = std::min(hi, b->user_high);
        }
        if (b->free_ends) {
            // The forward phase: Ties.LEFT over the pair as it is, Ties.RIGHT over both sequences reversed with each
            // sequence's free letters swapped end for end (reference tests/test_alignment.mojo:2054-2093). Its
            // band holds every diagonal a path may start or end on, and one either side.
            const bool right = b->options.right_ties;
            const int64_t e[4] = {right ? b->ends[1] : b->ends[0], right ? b->ends[0] : b->ends[1],
                                  right ? b->ends[3] : b->ends[2], right ? b->ends[2] : b->ends[3]};
            const int32_t f[4] = {(int32_t)std::min<int64_t>(e[0], n), (int32_t)std::min<int64_t>(e[1], n),
                                  (int32_t)std::min<int64_t>(e[2], m), (int32_t)std::min<int64_t>(e[3], m)};
            for (int k = 0; k < 4; ++k) b->a_free[4 * s + k] = f[k];
            lo = std::max(std::min(-f[0], end - f[3]) - 1, -n - 1);
            hi = std::min(std::max(f[2], end + f[1]) + 1, m + 1);
        }
        b->first_low[s] = lo;
        b->first_high[s] = hi;
        // A pair whose start and end diagonals lie further apart than the widest band is left unswept (its status
        // stays unsettled).
        const int cls = first_class(b, s, std::max(hi - lo + 1, b->initial_width));
        if (cls != CLASS_TOO_WIDE) b->first_lists[cls].push_back((int32_t)s);
        // A walk's moves, 2 bits each in 64-bit words; the CIGAR text, at most two bytes a move.
        b->scratch_base[s] = scratch;
        if (b->kind == DINARA_BATCH_ALIGNMENTS) {
            scratch += 8 * (((int64_t)n + m) / 32 + 1);
            text += 2 * ((int64_t)n + m) + 2;
        }
    }
    b->scratch_base[slots] = scratch;
    std::vector<int32_t> first_all;
    b->first_offset.assign(CLASSES + 1, 0);
    for (int c = 0; c < CLASSES; ++c) {
        b->first_offset[c] = (int64_t)first_all.size();
        first_all.insert(first_all.end(), b->first_lists[c].begin(), b->first_lists[c].end());
    }
    b->first_offset[CLASSES] = (int64_t)first_all.size();
    if (first_all.empty()) first_all.push_back(0);  // every pair too wide: the device list still needs room
    // The batch's buffers in one block, as far as it goes; what a run grows is allocated apart.
    DeviceContext *ctx = b->ctx;
    Carve carve;
    std::optional<CarveScope> scope;
    if (!CarveScope::active()) {
        const size_t slot_bytes = 256 + 8 * CLASSES + (b->unit ? 20 * EDIT_BINS + 64 : 0) + (b->free_ends ? 48 : 0);
        b->region = ctx->take_region((size_t)padded * 4 + slots * slot_bytes + scratch + text + (64 << 10));
        if (b->region.base) {
            carve.base = b->region.base;
            carve.size = b->region.size;
            carve.image = b->region.image;
            carve.strict = false;
            scope.emplace(&carve);
        }
    }
    if (b->free_ends) {
        // The forward phase's lists and bands, uploaded again at each run (the anchored phase writes its own).
        b->a_first_low = b->first_low;
        b->a_first_high = b->first_high;
        b->a_first_all = first_all;
        b->a_first_offset = b->first_offset;
        b->a_rows = b->rows;
        b->a_cols = b->cols;
        b->a_at.assign(std::max<int64_t>(slots, 1), 0);
        const size_t cap = (size_t)std::max<int64_t>(slots, 1);
        if (!b->view_rows_d.reserve(cap * 4) || !b->view_cols_d.reserve(cap * 4) || !b->view_ref_at_d.reserve(cap * 4) ||
            !b->view_qry_at_d.reserve(cap * 4) || !b->free_d.reserve(cap * 16) || !b->end_row_d.reserve(cap * 4) ||
            !b->end_col_d.reserve(cap * 4))
            return DINARA_OUT_OF_MEMORY;
    }

    // Upload.
    if (!b->tape.upload(ctx, tape.get(), (size_t)padded * 4) ||
        !b->group_base.upload(ctx, gbase.data(), gbase.size() * 8) ||
        !b->group_ref_words.upload(ctx, gref.data(), gref.size() * 4) ||
        !b->rows_d.upload(ctx, b->rows.data(), std::max<int64_t>(slots, 1) * 4) ||
        !b->cols_d.upload(ctx, b->cols.data(), std::max<int64_t>(slots, 1) * 4) ||
        !b->first_low_d.upload(ctx, b->first_low.data(), std::max<int64_t>(slots, 1) * 4) ||
        !b->first_high_d.upload(ctx, b->first_high.data(), std::max<int64_t>(slots, 1) * 4) ||
        !b->want_low.reserve(std::max<int64_t>(slots, 1) * 4) || !b->want_high.reserve(std::max<int64_t>(slots, 1) * 4) ||
        !b->cost.reserve(std::max<int64_t>(slots, 1) * 4) || !b->status.reserve(std::max<int64_t>(slots, 1) * 4) ||
        !b->walk_low.reserve(std::max<int64_t>(slots, 1) * 4) ||
        !b->walk_class.reserve(std::max<int64_t>(slots, 1) * 4) ||
        !b->retry_lists.reserve((size_t)2 * CLASSES * std::max<int64_t>(slots, 1) * 4) ||
        !b->retry_counts.reserve(2 * CLASSES * 4) ||
        (!b->unit && !b->strip_retries.reserve((size_t)2 * std::max<int64_t>(slots, 1) * sizeof(int4))) ||
        !b->first_lists_d.upload(ctx, first_all.data(), std::max<size_t>(first_all.size(), 1) * 4) ||
        !b->walk_flags.reserve(std::max<int64_t>(slots, 1) * 8))
        return DINARA_OUT_OF_MEMORY;
    if (b->unit)
        if (const int64_t code = unit_lists(b)) return code;
    if (b->kind == DINARA_BATCH_ALIGNMENTS) {
        if (!b->cigar_scratch.reserve(std::max<int64_t>(scratch, 1)) ||
            !b->cigar_scratch_base.upload(ctx, b->scratch_base.data(), b->scratch_base.size() * 8) ||
            !b->cigars.reserve(std::max<int64_t>(text, 1)) || !b->cigar_used.reserve(8) ||
            !b->cigar_offset.reserve(std::max<int64_t>(slots, 1) * 8) ||
            !b->cigar_length.reserve(std::max<int64_t>(slots, 1) * 4))
            return DINARA_OUT_OF_MEMORY;
    }
    return carve.flush(ctx) ? 0 : DINARA_OUT_OF_MEMORY;
}

SweepArgs sweep_args(dinara_batch *b) {
    SweepArgs a{};
    a.tape.words = static_cast<const uint32_t *>(b->tape.ptr);
    a.tape.group_base = static_cast<const int64_t *>(b->group_base.ptr);
    a.tape.group_ref_words = static_cast<const int32_t *>(b->group_ref_words.ptr);
    a.tape.rows = static_cast<const int32_t *>(b->rows_d.ptr);
    a.tape.cols = static_cast<const int32_t *>(b->cols_d.ptr);
    a.tape.bits = b->bits;
    a.slots = (int)b->slot_pair.size();
    a.want_low = static_cast<int32_t *>(b->want_low.ptr);
    a.want_high = static_cast<int32_t *>(b->want_high.ptr);
    a.costs = b->costs;
    a.strict = b->kind == DINARA_BATCH_ALIGNMENTS;
    a.cap = b->options.max_cost >= 0 ? b->options.max_cost : INT64_MAX / 4;
    a.user_band = b->user_band;
    a.user_low = b->user_low;
    a.user_high = b->user_high;
    a.eqx = b->options.eqx;
    a.forward_cigar = b->kind == DINARA_BATCH_ALIGNMENTS && !b->options.right_ties;
    a.record = b->kind == DINARA_BATCH_ALIGNMENTS;
    a.lds_limit = (int)b->lds_limit;
    a.cost = static_cast<int32_t *>(b->cost.ptr);
    a.status = static_cast<int32_t *>(b->status.ptr);
    a.walk_low = static_cast<int32_t *>(b->walk_low.ptr);
    a.walk_class = static_cast<int32_t *>(b->walk_class.ptr);
    a.walk_flags = static_cast<uint64_t *>(b->walk_flags.ptr);
    a.doubling = b->doubling ? 1 : 0;
    a.group16_top = b->group16_top;
    a.limits = b->limits;
    a.cigar_scratch = static_cast<char *>(b->cigar_scratch.ptr);
    a.cigar_scratch_base = static_cast<const int64_t *>(b->cigar_scratch_base.ptr);
    a.cigars = static_cast<char *>(b->cigars.ptr);
    a.cigar_used = static_cast<unsigned long long *>(b->cigar_used.ptr);
    a.cigar_offset = static_cast<int64_t *>(b->cigar_offset.ptr);
    a.cigar_length = static_cast<int32_t *>(b->cigar_length.ptr);
    a.retry_capacity = (int)std::max<size_t>(b->slot_pair.size(), 1);
    a.free_ends = b->free_ends ? 1 : 0;
    if (b->free_ends) {
        // The forward phase reads the pair as Ties.RIGHT's mirror or as it is; the anchored phase the other way,
        // as a global alignment's tape is (reference lanes.mojo:1523-1525).
        const bool right = b->options.right_ties;
        a.view_reversed = b->phase == 2 ? !right : right;
        a.lowest_end = b->phase == 2;
        a.record = b->kind == DINARA_BATCH_ALIGNMENTS && b->phase == 2;
        a.view_rows = static_cast<const int32_t *>(b->view_rows_d.ptr);
        a.view_cols = static_cast<const int32_t *>(b->view_cols_d.ptr);
        a.view_ref_at = static_cast<const int32_t *>(b->view_ref_at_d.ptr);
        a.view_qry_at = static_cast<const int32_t *>(b->view_qry_at_d.ptr);
        a.free = static_cast<const int32_t *>(b->free_d.ptr);
        a.end_row = static_cast<int32_t *>(b->end_row_d.ptr);
        a.end_col = static_cast<int32_t *>(b->end_col_d.ptr);
    }
    return a;
}


// Launches class `cls` over `count` slots listed at `list` (device memory), the longest of `longest` letters, filing
// retries where `round` says. Each launch keeps its decisions in an arena of its own, a fixed stride a listed pair, until
// the walk; a launch whose arena would pass the budget is cut in pieces. `arena_index` counts the run's arenas.
int64_t launch_class(dinara_batch *b, const SweepArgs &round, int cls, const int32_t *list, int64_t count, int longest,
                     size_t &arena_index, hipStream_t stream) {
    SweepArgs a = round;
    a.cls = cls;
    const bool wave = class_is_wave(cls);
    a.group_letters = group_region(longest);
    if (longest > b->limits.group_letters) a.group16_top = 0;  // past the packed cells' bound
    const size_t lds = wave ? (size_t)std::min<int>(std::max(longest, 4), (int)b->lds_limit)
                            : (size_t)(a.group16_top > 0 && cls >= 1 ? 8 : 4) * a.group_letters;
    int64_t chunk = count;
    size_t stride = 0;
    if (a.record) {
        // The launch's longest pair bounds every pair's decisions: rows for a wave band, tiles of 32
        // anti-diagonals (16 bytes a diagonal pair) for a group's.
        const int64_t bytes = wave ? (int64_t)std::min<int>(b->max_rows, longest) * class_width(cls)
                                   : ((int64_t)longest / 32 + 1) * (class_width(cls) / 2) * 16;
        stride = ((size_t)bytes + 255) & ~size_t(255);
        chunk = std::max<int64_t>(1, (int64_t)std::min<size_t>(count, ARENA_BUDGET / std::max<size_t>(stride, 1)));
    }
    for (int64_t start = 0; start < count; start += chunk) {
        a.list = list + start;
        a.count = (int)std::min(chunk, count - start);
        if (a.record) {
            if (arena_index == b->arenas.size()) b->arenas.push_back(new DeviceBuffer());
            DeviceBuffer *arena = b->arenas[arena_index++];
            if (!arena->reserve(std::max<size_t>(stride * a.count, 256))) return DINARA_OUT_OF_MEMORY;
            a.arena = static_cast<uint8_t *>(arena->ptr);
            a.arena_stride = (int64_t)stride;
        }
        launch_sweep(a, lds, stream);
        if (hipGetLastError() != hipSuccess) return DINARA_OUT_OF_MEMORY;
        b->launches += 1;
        b->class_launches[cls] += 1;
        b->class_pairs[cls] += a.count;
    }
    return 0;
}

// The columns a lane of a pair's strips holds: the fewest that take its columns in one strip, for a short query; for
// a longer one, eight (half the strips and pipeline starts of four, and less of a row step spent outside the cells).
int strip_c(int64_t m) { return m <= strip_columns(2) ? 2 : m <= strip_columns(4) ? 4 : 8; }

// A round of few strips is as long as its longest pair's pipeline, and a strip of four columns a lane hands on sooner
// than twice the half of one of eight (its step is shorter, and so are its rows): up to this many strips of eight, four.
// A round that fills the chip pays for its cells. Four against eight, ms: uneven gap-affine pairs (1.5 kbp median, up to
// 20 kbp) 1,000 9.1 and 10.1, 4,000 12.9 and 13.2, 8,000 18.8 and 19.0, 200,000 251 and 236; two-piece CIGARs (1.5 kbp)
// 1,000 10.2 and 12.6, 4,000 19.5 and 19.5, 8,000 31 and 29. Gap-affine CIGARs, whose decisions of four columns go out
// in half lines, turn sooner: 500 21.5 and 22.0, 1,000 24.1 and 23.5, 2,000 29.0 and 26.6, 8,000 67 and 50.
constexpr int64_t FEW_STRIPS = 16384, FEW_STRIPS_ONE_PIECE_CIGARS = 4096;
// Whatever their number, strips of four where costs alone are kept and the band is narrower than this: a strip's rows
// are its band's and its columns'. 4,000 pairs of 3 kbp at 5% 4.4 -> 3.9 ms; their CIGARs 13.1 -> 16.5, so not those.
constexpr int NARROW_BAND = 512;

// A strip launch's parts: consecutive pairs of the plan whose decisions and carry records fit ARENA_BUDGET together. A
// round of costs keeps no decisions, but each pair's carry records (8 bytes a row a strip, 16 under two pieces; 0.8 MB
// for a pair of 10,000 letters in 4,500 diagonals), so what a batch asks for would grow with its pairs. A part costs its
// longest pair's pipeline once more: 200,000 uneven distances 241 ms in one part of 10 GB, 243 in parts of 4 GB, 269 in
// parts of 1 GB. DINARA_STRIP_BUDGET sets the bytes a part may take, for checking.
// A round's plan on the host, the context's: made anew for each round (under its lock), its memory kept while it is small.
struct StripPlan {
    std::vector<StripPair> pairs;
    std::vector<int2> order;  // of the parts with a pair of several strips
    std::vector<size_t> at;
};
constexpr size_t PLAN_KEPT = size_t(1) << 18;  // pairs, strips

StripPlan &strip_plan_of(DeviceContext *ctx) {
    if (!ctx->strip_plan) ctx->strip_plan = new StripPlan();
    return *static_cast<StripPlan *>(ctx->strip_plan);
}

// The plan of the pairs listed in `bands` (slot, low, high): each pair's strips, where its records lie, and the order
// its strips are claimed in: the strips furthest from their pair's end first, so that the longest pipelines start first
// and a strip always follows the one to its left. `round`: a round of bands, whose strips may be narrower.
StripParts plan_strips(const dinara_batch *b, const std::vector<int4> &bands, bool record, bool round) {
    StripPlan &plan = strip_plan_of(b->ctx);
    StripParts out;
    plan.pairs.clear();
    plan.order.clear();
    // A large round's memory goes when the next is planned (this one's is read by upload_strips until then).
    if (plan.pairs.capacity() > PLAN_KEPT) std::vector<StripPair>().swap(plan.pairs);
    if (plan.order.capacity() > PLAN_KEPT) std::vector<int2>().swap(plan.order);
    plan.pairs.reserve(bands.size());
    std::vector<size_t> &at = plan.at;
    const int pieces = b->costs.pieces == 2 ? 2 : 1;
    const bool views = b->free_ends;
    int widest_c = 8, narrow_c = round && !record ? 4 : 8;
    if (const char *set = std::getenv("DINARA_STRIP_COLUMNS")) {  // for checking: 2, 4 or 8 at most
        widest_c = narrow_c = std::strtol(set, nullptr, 10) <= 2 ? 2 : std::strtol(set, nullptr, 10) <= 4 ? 4 : 8;
    } else if (round) {
        int64_t strips = 0;
        for (const int4 &band : bands) strips += b->cols[band.x] / strip_columns(8) + 1;
        if (strips <= (record && pieces == 1 ? FEW_STRIPS_ONE_PIECE_CIGARS : FEW_STRIPS)) widest_c = narrow_c = 4;
    }
    size_t budget = ARENA_BUDGET;
    if (const char *set = std::getenv("DINARA_STRIP_BUDGET")) budget = std::strtoull(set, nullptr, 10);
    for (size_t next = 0; next < bands.size();) {
        StripPart part{plan.pairs.size(), 0, plan.order.size(), 0, 0, 0};
        int most = 0;
        for (; next < bands.size(); ++next) {
            const int4 &band = bands[next];
            const int64_t n = views && b->phase == 2 ? b->b_rows_h[band.x] : b->rows[band.x];
            const int64_t m = views && b->phase == 2 ? b->b_cols_h[band.x] : b->cols[band.x];
            StripPair p{};
            p.slot = band.x;
            p.lo = band.y;
            p.hi = band.z;
            p.c = std::min(strip_c(m), p.hi - p.lo + 1 < NARROW_BAND ? narrow_c : widest_c);
            p.strips = (int)std::max<int64_t>(1, (m + strip_columns(p.c) - 1) / strip_columns(p.c));
            p.rows = (int)std::max<int64_t>(1, std::min<int64_t>(n, (int64_t)p.hi - p.lo + strip_columns(p.c)));
            const size_t records = (size_t)p.strips * p.rows * 64;
            const size_t bytes = record ? (records * strip_record_bytes(p.c, pieces) + 255) & ~size_t(255) : 0;
            const size_t carried = p.strips > 1 ? (size_t)p.strips * p.rows * pieces : 0;
            const size_t carry_bytes = 8 * (part.carry_words + carried);
            if (part.pairs > 0 && part.decision_bytes + bytes + carry_bytes > budget) break;
            p.decision_at = (int64_t)part.decision_bytes;
            p.carry_at = (int64_t)part.carry_words;
            part.decision_bytes += bytes;
            part.carry_words += carried;
            part.strips += p.strips;
            ++part.pairs;
            most = std::max(most, p.strips);
            plan.pairs.push_back(p);
            const int cls = band_class(p.hi - p.lo + 1, 1, false, BandLimits{0, 0, 0, 0, 0, 1, 1 << 20});
            out.class_pairs[std::max(CLASS_STRIP_FIRST, cls)] += 1;
        }
        out.decision_bytes = std::max(out.decision_bytes, part.decision_bytes);
        out.carry_words = std::max(out.carry_words, part.carry_words);
        out.parts.push_back(part);
        if (most == 1) continue;  // a strip a pair, claimed as they are listed
        // By strips left to the pair's end, most first.
        at.assign((size_t)most + 1, 0);
        for (size_t i = 0; i < part.pairs; ++i)
            for (int left = 1; left <= plan.pairs[part.pair + i].strips; ++left) ++at[most - left];
        for (size_t k = 0, sum = 0; k < at.size(); ++k) {
            const size_t here = at[k];
            at[k] = sum;
            sum += here;
        }
        plan.order.resize(part.strip + part.strips);
        for (size_t i = 0; i < part.pairs; ++i) {
            const int strips = plan.pairs[part.pair + i].strips;
            for (int strip = 0; strip < strips; ++strip)
                plan.order[part.strip + at[most - (strips - strip)]++] = make_int2((int)i, strip);
        }
    }
    out.pairs = plan.pairs.size();
    return out;
}

// Room for the launches of a plan's parts.
bool reserve_strips(dinara_batch *b, const StripParts &of) {
    size_t most = 1;
    for (const StripPart &part : of.parts) most = std::max(most, part.pairs);
    return b->strip_counts.reserve((most + 1) * 4) && b->strip_best.reserve(most * 8) &&
           b->strip_carry.reserve(std::max<size_t>(of.carry_words, 1) * 8) &&
           (of.decision_bytes == 0 || b->strip_decisions.reserve(of.decision_bytes));
}

// The plan made last onto the device: its pairs, then its order. Waits for the main stream.
bool upload_strips(dinara_batch *b, DeviceBuffer &to) {
    const StripPlan &plan = strip_plan_of(b->ctx);
    const size_t pairs = plan.pairs.size() * sizeof(StripPair), order = plan.order.size() * sizeof(int2);
    hipStream_t stream = b->ctx->stream;
    return to.reserve(pairs + order) &&
           hipMemcpyAsync(to.ptr, plan.pairs.data(), pairs, hipMemcpyHostToDevice, stream) == hipSuccess &&
           (order == 0 || hipMemcpyAsync(static_cast<uint8_t *>(to.ptr) + pairs, plan.order.data(), order,
                                         hipMemcpyHostToDevice, stream) == hipSuccess) &&
           hipStreamSynchronize(stream) == hipSuccess;
}

// Where among a round's counts its strips' expired waits are (strip classes are counted together at the first).
constexpr int STRIP_EXPIRED = CLASS_STRIP_FIRST + 1;

// The polls of a round's waits; DINARA_STRIP_POLLS sets them, for checking.
int strip_polls() {
    const char *set = std::getenv("DINARA_STRIP_POLLS");
    return set ? (int)std::strtol(set, nullptr, 10) : STRIP_POLL_LIMIT;
}

// The launches of a plan (on the device at `plan`) on `stream`, each part's sweep and (when decisions are kept) its walks,
// filing unproven pairs where `round` says; `whole`: the bands are whole matrices.
int64_t launch_strips(dinara_batch *b, const SweepArgs &round, const StripParts &of, const DeviceBuffer &plan, bool whole,
                      hipStream_t stream) {
    const StripPair *pairs = static_cast<const StripPair *>(plan.ptr);
    for (const StripPart &part : of.parts) {
        StripArgs a{};
        a.s = round;
        a.pairs = pairs + part.pair;
        a.order = part.strips == part.pairs ? nullptr : reinterpret_cast<const int2 *>(pairs + of.pairs) + part.strip;
        a.count = (int)part.pairs;
        a.strips = (int)part.strips;
        a.whole = whole ? 1 : 0;
        a.decisions = part.decision_bytes ? static_cast<uint8_t *>(b->strip_decisions.ptr) : nullptr;
        a.carry = static_cast<unsigned long long *>(b->strip_carry.ptr);
        a.claim = static_cast<int *>(b->strip_counts.ptr);
        a.done = a.claim + 1;
        a.polls = whole ? STRIP_POLL_LIMIT : strip_polls();
        a.expired = whole ? nullptr : round.retry_counts + STRIP_EXPIRED;
        a.best = static_cast<unsigned long long *>(b->strip_best.ptr);
        if (hipMemsetAsync(b->strip_counts.ptr, 0, (part.pairs + 1) * 4, stream) != hipSuccess ||
            (part.carry_words &&
             hipMemsetAsync(b->strip_carry.ptr, 0, part.carry_words * 8, stream) != hipSuccess) ||
            (b->free_ends && hipMemsetAsync(b->strip_best.ptr, 0xFF, part.pairs * 8, stream) != hipSuccess))
            return DINARA_OUT_OF_MEMORY;
        launch_strip_sweep(a, stream);
        if (a.decisions) launch_strip_walk(a, stream);
        if (hipPeekAtLastError() != hipSuccess) return DINARA_OUT_OF_MEMORY;
        b->launches += 1;
    }
    return 0;
}

// ------------------------------------------------------------------ the unit-cost path

// The unit path's first queues: each pair in the narrowest bin of the first pass's set that holds its first band,
// no narrower than its length class's start bin (under band doubling, the first such bin of any set whose width is a
// power of two), placed around the start and end diagonals. Caller holds the device lock.
int64_t unit_lists(dinara_batch *b) {
    const int64_t slots = (int64_t)b->slot_pair.size();
    const size_t cap = (size_t)std::max<int64_t>(slots, 1);
    std::vector<int32_t> lists(EDIT_BINS * cap, 0), counts(EDIT_BINS, 0);
    b->edit_first_low.assign(cap, 0);
    b->edit_first_bin.assign(cap, -1);
    int64_t first_count[EDIT_BINS] = {}, retry_reach[EDIT_BINS] = {}, trace_reach[EDIT_BINS] = {};
    for (int64_t s = 0; s < slots; ++s) {
        const int n = b->rows[s], m = b->cols[s];
        const int lo = b->first_low[s], hi = b->first_high[s];
        const int from = b->start_bin[edit_length_class(std::max(n, m))];
        // A band placed inside the matrix's diagonals and n + m + 3 wide proves any pair, and no traced band is
        // wider than n + m + 1: the bins a pair can reach.
        const int widest = edit_widest(n + m);
        const int bin = b->doubling ? edit_power_bin_for(hi - lo + 1, from)
                                    : edit_first_bin(hi - lo + 1, from, b->first_bins, std::max(from, widest));
        if (bin < 0) continue;  // wider than the widest band: left unsettled
        b->edit_first_low[s] = edit_place(lo, hi, edit_width(bin), n, m);
        b->edit_first_bin[s] = bin;
        lists[bin * cap + counts[bin]++] = (int32_t)s;
        ++first_count[bin];
        for (int k = bin + 1; k <= widest; ++k) ++retry_reach[k];
        for (int k = 0; k <= widest; ++k) ++trace_reach[k];
    }
    bool same_reach = true;
    for (int k = 0; k < EDIT_BINS; ++k) {
        same_reach = same_reach && first_count[k] == b->first_count[k] && retry_reach[k] == b->retry_reach[k] &&
                     trace_reach[k] == b->trace_reach[k];
        b->first_count[k] = first_count[k];
        b->retry_reach[k] = retry_reach[k];
        b->trace_reach[k] = trace_reach[k];
    }
    b->seeded_start[0] = -1;  // host-filed queues: the device seeding's shape no longer holds
    if (!same_reach && b->edit_graph) {  // the launches' shape changes
        (void)hipGraphExecDestroy(b->edit_graph);
        b->edit_graph = nullptr;
    }
    // The captured graph reads these buffers where they were: it is kept unless one moves.
    DeviceBuffer *held[] = {&b->edit_first_lists, &b->edit_first_counts, &b->edit_first_low_d, &b->edit_band_low,
                            &b->edit_lists, &b->edit_counts, &b->edit_retry_lists, &b->edit_retry_counts,
                            &b->edit_later_lists, &b->edit_later_counts, &b->trace_lists, &b->trace_counts, &b->trace_offset,
                            &b->walk_ready, &b->walk_moves, &b->walk_early, &b->deferred, &b->deferred_count, &b->deferred_held,
                            &b->arena_used, &b->edit_stats, &b->edit_work};
    void *before[sizeof(held) / sizeof(held[0])];
    for (size_t i = 0; i < sizeof(held) / sizeof(held[0]); ++i) before[i] = held[i]->ptr;
    const int64_t code = unit_buffers(b, lists, counts, cap);
    for (size_t i = 0; i < sizeof(held) / sizeof(held[0]); ++i)
        if (held[i]->ptr != before[i] && b->edit_graph) {
            (void)hipGraphExecDestroy(b->edit_graph);
            b->edit_graph = nullptr;
        }
    return code;
}

int64_t unit_buffers(dinara_batch *b, const std::vector<int32_t> &lists, const std::vector<int32_t> &counts,
                     size_t cap) {
    DeviceContext *ctx = b->ctx;
    if (!b->edit_first_lists.upload(ctx, lists.data(), lists.size() * 4) ||
        !b->edit_first_counts.upload(ctx, counts.data(), counts.size() * 4) ||
        !b->edit_first_low_d.upload(ctx, b->edit_first_low.data(), cap * 4) || !b->edit_band_low.reserve(cap * 4) ||
        !b->edit_lists.reserve(EDIT_BINS * cap * 4) || !b->edit_counts.reserve(2 * EDIT_BINS * 4) ||
        !b->edit_retry_lists.reserve(EDIT_BINS * cap * 4) || !b->edit_retry_counts.reserve(2 * EDIT_BINS * 4) ||
        !b->edit_later_lists.reserve(EDIT_BINS * cap * 4) || !b->edit_later_counts.reserve(3 * EDIT_BINS * 4) ||
        !b->trace_lists.reserve(EDIT_BINS * cap * 4) || !b->trace_counts.reserve(2 * EDIT_BINS * 4) ||
        !b->trace_offset.reserve(cap * 8) || !b->walk_ready.reserve(cap * 4) ||
        !b->walk_moves.reserve(cap * 4) || !b->walk_early.reserve(cap * 4) ||
        !b->deferred.reserve(cap * 4) || !b->deferred_count.reserve(4) || !b->deferred_held.reserve(cap * 4) ||
        !b->arena_used.reserve(8) || !b->edit_stats.reserve((2 * EDIT_BINS + 2) * 4) ||
        !b->edit_work.reserve(2 * EDIT_BINS * 8))
        return DINARA_OUT_OF_MEMORY;
    return 0;
}

EditArgs edit_args(dinara_batch *b) {
    EditArgs e{};
    e.s = sweep_args(b);
    // The certificate and the cap in unit terms: every cost is `unit_scale` times the unit cost.
    e.s.costs = CostParams{1, 0, 1, 0, 1, 1, 1, 1, 0, 1, 0, 1, 1, 1};
    e.s.cap = b->options.max_cost >= 0 ? b->options.max_cost / b->unit_scale : INT64_MAX / 4;
    e.scale = b->unit_scale;
    e.capacity = (int)std::max<size_t>(b->slot_pair.size(), 1);
    e.band_low = static_cast<int32_t *>(b->edit_band_low.ptr);
    e.first_band_low = static_cast<const int32_t *>(b->edit_first_low_d.ptr);
    e.lists = static_cast<int32_t *>(b->edit_lists.ptr);
    e.counts = static_cast<int32_t *>(b->edit_counts.ptr);
    e.file_lists = static_cast<int32_t *>(b->edit_retry_lists.ptr);
    e.file_counts = static_cast<int32_t *>(b->edit_retry_counts.ptr);
    e.spare_counts = static_cast<int32_t *>(b->edit_later_counts.ptr);
    e.first_lists = static_cast<int32_t *>(b->edit_first_lists.ptr);
    e.first_counts = static_cast<const int32_t *>(b->edit_first_counts.ptr);
    e.first_counts_out = static_cast<int32_t *>(b->edit_first_counts.ptr);
    e.first_low_out = static_cast<int32_t *>(b->edit_first_low_d.ptr);
    e.trace_lists = static_cast<int32_t *>(b->trace_lists.ptr);
    e.trace_counts = static_cast<int32_t *>(b->trace_counts.ptr);
    e.trace_offset = static_cast<int64_t *>(b->trace_offset.ptr);
    e.walk_ready = static_cast<int32_t *>(b->walk_ready.ptr);
    e.walk_moves = static_cast<int32_t *>(b->walk_moves.ptr);
    e.walk_early = static_cast<int32_t *>(b->walk_early.ptr);
    e.deferred = static_cast<int32_t *>(b->deferred.ptr);
    e.deferred_count = static_cast<int32_t *>(b->deferred_count.ptr);
    e.arena = static_cast<uint8_t *>(const_cast<void *>(b->arena_ptr));
    e.arena_used = static_cast<unsigned long long *>(b->arena_used.ptr);
    e.arena_capacity = b->arena_capacity;
    e.stats = static_cast<uint32_t *>(b->edit_stats.ptr);
    e.work = static_cast<unsigned long long *>(b->edit_work.ptr);
    e.one_pair = b->persistent ? 0 : 1;
    e.keep_first = b->keep_first && b->kind == DINARA_BATCH_ALIGNMENTS ? 1 : 0;
    return e;
}

// The slots walked a wave a pair: those whose longer side is at least EDIT_WALK_LONG letters, the first ones (slots
// are longest first).
int long_walks(const dinara_batch *b) {
    int count = 0;
    while (count < (int)b->rows.size() && std::max(b->rows[count], b->cols[count]) >= EDIT_WALK_LONG) ++count;
    return count;
}

// The walk of every slot ready for it: the long slots on `aside` and the others on `stream` at once (forked and joined
// by marks `mark` and `mark` + 1; `mark` + 2 marks both ended; one after the other when `aside` is `stream`), then
// the CIGAR text on `stream`.
void walk_slots(dinara_batch *b, const EditArgs &a, hipStream_t stream, hipStream_t aside, int mark, bool early) {
    DeviceContext *ctx = b->ctx;
    const int slots = (int)b->slot_pair.size(), longs = long_walks(b);
    if (longs > 0 && aside == stream) {
        launch_edit_walk_long(a, longs, stream, early);
    } else if (longs > 0) {
        (void)hipEventRecord(ctx->mark(mark), stream);
        (void)hipStreamWaitEvent(aside, ctx->mark(mark), 0);
        launch_edit_walk_long(a, longs, aside, early);
        (void)hipEventRecord(ctx->mark(mark + 1), aside);
    }
    launch_edit_walk_short(a, longs, slots, stream, early);
    if (longs > 0 && aside != stream) (void)hipStreamWaitEvent(stream, ctx->mark(mark + 1), 0);
    (void)hipEventRecord(ctx->mark(mark + 2), stream);
    launch_edit_text(a, slots, stream, early);
}

// Workgroups of a bin's launch that may meet `reach` pairs: enough for every one at once, at most `grid_per_cu` a
// compute unit when the groups refill from the queue; 0 when it meets none.
int edit_grid(const dinara_batch *b, int bin, int64_t reach) {
    if (reach == 0) return 0;
    const int64_t every = (reach * edit_lanes(bin) + 255) / 256;
    if (!b->persistent) return (int)std::max<int64_t>(1, every);
    return (int)std::max<int64_t>(1, std::min<int64_t>(every, (int64_t)b->ctx->compute_units * b->grid_per_cu));
}

// The arena the kept bands' decisions may take (`bound`: no band is wider than its whole matrix) and what the batch is
// likely to need (`ask`: bands a quarter of the pairs' longer side). Mapping device memory takes about 30 ms a GB, and
// 20,000 uneven pairs are bound by the 0.6 of the card's memory a run may take: a process's first run on such a batch
// spent 5.1 s there, and so did every later batch whose bound came out a little larger. So the arena is made for what
// is likely, kept, and doubled when a run has left pairs without room (they are traced in further passes). At most 0.6
// of the free memory, at least 1 MiB; DINARA_TRACE_ARENA sets it in bytes.
struct ArenaNeed {
    size_t ask, bound;
};
ArenaNeed arena_need(const dinara_batch *b) {
    if (const char *env = std::getenv("DINARA_TRACE_ARENA")) {
        const size_t set = std::max<size_t>(std::strtoull(env, nullptr, 10), 4096);
        return {set, set};
    }
    size_t bound = 0, likely = 0;
    for (size_t s = 0; s < b->slot_pair.size(); ++s) {
        const int n = b->rows[s], m = b->cols[s], widest = edit_widest(n + m);
        const int usual = edit_bin_for(std::abs(m - n) + std::max(n, m) / 4 + 64, 0);
        bound += (size_t)edit_trace_bytes(m, widest);
        likely += (size_t)edit_trace_bytes(m, usual < 0 ? widest : std::min(usual, widest));
    }
    size_t free_bytes = 0, total = 0;
    (void)hipMemGetInfo(&free_bytes, &total);
    if (b->ctx->edit_arena) free_bytes += b->ctx->edit_arena->size;  // the arena itself is there to be used
    const size_t most = std::max<size_t>(free_bytes / 10 * 6, size_t(1) << 20);
    if (b->keep_first) bound *= 3;  // every attempt keeps its decisions
    bound = std::min(std::max<size_t>(bound, size_t(1) << 20), most);
    return {std::min(bound, std::max<size_t>(likely, size_t(1) << 31)), bound};
}

// The streams a round of band sweeps runs on: the main one and three at its side, HIP's hardware queues by default.
constexpr int SWEEP_STREAMS = 4;

// Timing events of a run launched kernel by kernel: a pair for each bin's first sweep, retry sweep and tracing
// sweep (the bins that share a launch share bin 0's pair), and for the walk.
constexpr int EV_FIRST = 0, EV_RETRY = 2 * EDIT_BINS, EV_TRACE = 4 * EDIT_BINS, EV_WALK = 6 * EDIT_BINS;
// Marks (untimed events) that order the streams: a pass's fork and its wide bins' ends (each pass WIDE_BINS + 1), the
// fork and join of what runs beside the retries, and the walks' (the early walk's three, the last walk's three).
constexpr int WIDE_BINS = EDIT_BINS - EDIT_NARROW;
constexpr int FIRST_MARKS = 0, RETRY_MARKS = FIRST_MARKS + WIDE_BINS + 1, TRACE_MARKS = RETRY_MARKS + WIDE_BINS + 1,
              BESIDE_MARKS = TRACE_MARKS + WIDE_BINS + 1, WALK_MARKS = BESIDE_MARKS + 2;
// The side streams: one a wide bin (the first walks the long pairs once the sweeps are done), one for what runs beside
// the retries. With the main stream they are four, as many as HIP's hardware queues by default: streams sharing a queue
// run one after the other.
constexpr int SIDE_WIDE = 0, SIDE_BESIDE = WIDE_BINS;

int timing_pair(const dinara_batch *b, int bin) { return b->side_by_side_bins && bin < EDIT_NARROW ? 0 : 2 * bin; }

// One sweep of every bin's queue (`reach`: the pairs each may hold): the one-word bins in one launch on `stream`, the
// wider ones beside it on streams forked from the main one, widest first (their pairs are the longest chains); or, not
// side by side, the bins one after another on `stream`. `mark` is the first of the pass's marks; `timed` records the
// pairs of events from `ev`. The main stream waits for the wider bins at join_bins, whatever `stream` is: under capture
// every fork must come from the stream that captures and every join go to it. A stream forked from one stream and
// joined to another that was itself forked leaves each the other's parent, and with HIP 7.0 (as shipped with PyTorch)
// ending such a capture, whose streams end their children's first, ended the process.
void sweep_bins(dinara_batch *b, const EditArgs &a, bool trace, const int64_t (&reach)[EDIT_BINS], hipStream_t stream,
                int mark, bool timed, int ev) {
    DeviceContext *ctx = b->ctx;
    const auto around = [&](int pair, hipStream_t on, auto launch) {
        if (timed) (void)hipEventRecord(ctx->event(ev + pair), on);
        launch();
        if (timed) (void)hipEventRecord(ctx->event(ev + pair + 1), on);
        b->launches += 1;
    };
    int grid[EDIT_BINS], narrow = 0;
    for (int bin = 0; bin < EDIT_BINS; ++bin) {
        grid[bin] = edit_grid(b, bin, reach[bin]);
        if (bin < EDIT_NARROW) narrow += grid[bin];
    }
    if (!b->side_by_side_bins) {
        for (int bin = 0; bin < EDIT_BINS; ++bin) {
            if (!grid[bin]) continue;
            int only[EDIT_BINS] = {};
            only[bin] = grid[bin];
            around(2 * bin, stream, [&] {
                if (bin < EDIT_NARROW) launch_edit_sweep(a, trace, only, stream);
                else launch_edit_sweep_wide(a, bin, trace, grid[bin], stream);
            });
        }
        return;
    }
    bool forked = false;
    for (int bin = EDIT_BINS - 1; bin >= EDIT_NARROW; --bin) {
        if (!grid[bin]) continue;
        hipStream_t side = stream;
        if (!b->one_stream) {
            if (!forked) (void)hipEventRecord(ctx->mark(mark), ctx->stream);
            forked = true;
            side = ctx->side(SIDE_WIDE + bin - EDIT_NARROW);
            (void)hipStreamWaitEvent(side, ctx->mark(mark), 0);
        }
        around(2 * bin, side, [&] { launch_edit_sweep_wide(a, bin, trace, grid[bin], side); });
        if (!b->one_stream) (void)hipEventRecord(ctx->mark(mark + 1 + bin - EDIT_NARROW), side);
    }
    if (narrow) around(0, stream, [&] { launch_edit_sweep(a, trace, grid, stream); });
}

// The main stream waits for the wider bins of the pass whose marks start at `mark`.
void join_bins(dinara_batch *b, const int64_t (&reach)[EDIT_BINS], int mark) {
    if (!b->side_by_side_bins || b->one_stream) return;
    for (int bin = EDIT_NARROW; bin < EDIT_BINS; ++bin)
        if (edit_grid(b, bin, reach[bin]))
            (void)hipStreamWaitEvent(b->ctx->stream, b->ctx->mark(mark + 1 + bin - EDIT_NARROW), 0);
}

// The run's launches: reset; every bin's first queue; the retry queues; then (alignments) the tracing sweep, and the
// walk. `timed` records an event pair around each launch (not under capture).
//
// Under the certified policy a retry always proves its pair: its band holds every diagonal a path cheaper than the
// first band's cost could visit, its own cost is no higher, so no path outside it is cheaper (certify). So there are no
// later retries, and an alignment's retries keep their decisions (a band traced again would cost a long pair's chain
// twice), while the pairs the first pass proved are traced beside them. 4,000 uneven pairs, one call, the tracing pass
// after the retries: 42.3 ms; beside them and every bin in one launch: 17.1 ms. Plain band doubling files again and
// again: its later retries go one bin after another, and its tracing sweep follows them.
//
// With kept first bands the tracing queues stay empty: a pair whose decisions found no room is deferred (the arena's
// used count has then passed its capacity for the whole run), not queued.
int64_t enqueue_unit(dinara_batch *b, const EditArgs &a, bool timed, bool trace) {
    DeviceContext *ctx = b->ctx;
    const int slots = (int)b->slot_pair.size();
    launch_edit_reset(a, slots, ctx->stream);
    sweep_bins(b, a, false, b->first_count, ctx->stream, FIRST_MARKS, timed, EV_FIRST);
    join_bins(b, b->first_count, FIRST_MARKS);
    // Kept decisions: the pairs the first pass proved are walked on a stream of their own while the retries sweep.
    const bool early = trace && b->keep_first;
    const bool beside = trace && !b->keep_first && !b->doubling;
    if (early) {
        launch_edit_snapshot(a, slots, ctx->stream);
        (void)hipEventRecord(ctx->mark(BESIDE_MARKS), ctx->stream);
        hipStream_t walker = ctx->side(SIDE_BESIDE);
        (void)hipStreamWaitEvent(walker, ctx->mark(BESIDE_MARKS), 0);
        // The early walk's two launches one after the other: side by side they slow the retries beside them,
        // whose long pairs are the run's tail.
        walk_slots(b, a, walker, walker, WALK_MARKS, true);
        (void)hipEventRecord(ctx->mark(BESIDE_MARKS + 1), walker);
    }
    EditArgs retry = a;
    retry.lists = a.file_lists;
    retry.counts = a.file_counts;
    retry.file_lists = static_cast<int32_t *>(b->edit_later_lists.ptr);
    retry.file_counts = static_cast<int32_t *>(b->edit_later_counts.ptr);
    if (beside) {
        retry.keep_first = 1;
        (void)hipEventRecord(ctx->mark(BESIDE_MARKS), ctx->stream);
        hipStream_t tracer = ctx->side(SIDE_BESIDE);
        (void)hipStreamWaitEvent(tracer, ctx->mark(BESIDE_MARKS), 0);
        sweep_bins(b, a, true, b->trace_reach, tracer, TRACE_MARKS, timed, EV_TRACE);
        (void)hipEventRecord(ctx->mark(BESIDE_MARKS + 1), tracer);
    }
    sweep_bins(b, retry, false, b->retry_reach, ctx->stream, RETRY_MARKS, timed, EV_RETRY);
    join_bins(b, b->retry_reach, RETRY_MARKS);
    if (b->doubling) {
        EditArgs later = retry;
        later.lists = retry.file_lists;
        later.counts = retry.file_counts;
        for (int bin = 0; bin < EDIT_BINS; ++bin) {
            if (!edit_power_bin(bin)) continue;
            int64_t only[EDIT_BINS] = {};
            only[bin] = b->retry_reach[bin];
            sweep_bins(b, later, false, only, ctx->stream, RETRY_MARKS, false, 0);
            join_bins(b, only, RETRY_MARKS);
        }
    }
    if (trace) {
        if (!b->keep_first && b->doubling)
            sweep_bins(b, a, true, b->trace_reach, ctx->stream, TRACE_MARKS, timed, EV_TRACE);
        if (!b->keep_first) join_bins(b, b->trace_reach, TRACE_MARKS);
        if (beside) (void)hipStreamWaitEvent(ctx->stream, ctx->mark(BESIDE_MARKS + 1), 0);
        // The last walk follows the early walk's kernels (it writes moves of slots the early walk marked unwalked)
        // and runs while the early walk's text is made; the run ends when both texts are made.
        if (early) (void)hipStreamWaitEvent(ctx->stream, ctx->mark(WALK_MARKS + 2), 0);
        if (timed) (void)hipEventRecord(ctx->event(EV_WALK), ctx->stream);
        walk_slots(b, a, ctx->stream, ctx->side(SIDE_WIDE), WALK_MARKS + 3, false);
        if (timed) (void)hipEventRecord(ctx->event(EV_WALK + 1), ctx->stream);
        if (early) (void)hipStreamWaitEvent(ctx->stream, ctx->mark(BESIDE_MARKS + 1), 0);
    }
    return hipPeekAtLastError() == hipSuccess ? 0 : DINARA_OUT_OF_MEMORY;
}

// The unit-cost run: one captured graph (or the same launches one by one, timed), then further tracing passes for
// pairs the arena had no room for. `trace` false skips the tracing (the autotuner's runs).
int64_t run_unit(dinara_batch *b, bool trace) {
    DeviceContext *ctx = b->ctx;
    const int64_t slots = (int64_t)b->slot_pair.size();
    trace = trace && b->kind == DINARA_BATCH_ALIGNMENTS;
    b->launches = b->first_proven = b->graph_used = b->trace_passes = 0;
    b->run_ms = b->sweep_ms = b->walk_ms = 0;
    for (int bin = 0; bin < EDIT_BINS; ++bin) b->edit_ms[bin] = b->trace_ms[bin] = b->edit_sweeps[bin] = b->trace_sweeps[bin] = 0;
    if (slots == 0) {
        b->ran = true;
        return 0;
    }
    if (b->kind == DINARA_BATCH_ALIGNMENTS) {
        // The context's arena, grown when this batch is likely to need more than it holds (by half at least, so that
        // a run of ever larger batches maps it a few times only) or the last run had too little; the graph is made
        // again when the arena it was captured with moved or this batch's share of it changed.
        if (!ctx->edit_arena) ctx->edit_arena = new DeviceBuffer();
        if (!b->arena_bound) {
            const ArenaNeed need = arena_need(b);
            b->arena_ask = need.ask;
            b->arena_bound = need.bound;
        }
        const size_t held = ctx->edit_arena->size, ask = std::min(std::max(b->arena_ask, ctx->arena_wanted), b->arena_bound);
        if (held < ask) {
            // Not past the memory there is now (the bound is the batch's first run's): a smaller arena serves with
            // more passes, so what cannot be had is not asked for again, and the size held before is taken back.
            size_t free_bytes = 0, total = 0;
            (void)hipMemGetInfo(&free_bytes, &total);
            if (held == 0 || ask - held <= free_bytes) {
                ctx->edit_arena->release();
                if (!ctx->edit_arena->reserve(std::min(std::max(ask, held + held / 2), b->arena_bound)) &&
                    !ctx->edit_arena->reserve(ask)) {
                    size_t less = std::max(held, ask / 2);
                    while (!ctx->edit_arena->reserve(less)) {
                        if (less <= (size_t(1) << 20)) return DINARA_OUT_OF_MEMORY;
                        less /= 2;
                    }
                }
            }
            if (ctx->edit_arena->size < ask) {
                b->arena_ask = std::min(b->arena_ask, ctx->edit_arena->size);
                ctx->arena_wanted = 0;
            }
        }
        const size_t bytes = std::min(ctx->edit_arena->size, b->arena_bound);
        if (b->arena_ptr != ctx->edit_arena->ptr || b->arena_capacity != bytes) {
            b->arena_ptr = ctx->edit_arena->ptr;
            b->arena_capacity = bytes;
            if (b->edit_graph) {
                (void)hipGraphExecDestroy(b->edit_graph);
                b->edit_graph = nullptr;
            }
        }
    }
    const EditArgs a = edit_args(b);
    const bool graph = b->use_graph && trace == (b->kind == DINARA_BATCH_ALIGNMENTS);
    if (graph) {
        if (!b->edit_graph) {
            hipGraph_t captured = nullptr;
            if (hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal) != hipSuccess)
                return DINARA_OUT_OF_MEMORY;
            const int64_t code = enqueue_unit(b, a, false, trace);
            const hipError_t ended = hipStreamEndCapture(ctx->stream, &captured);
            if (code || ended != hipSuccess) return DINARA_OUT_OF_MEMORY;
            const hipError_t made = hipGraphInstantiate(&b->edit_graph, captured, nullptr, nullptr, 0);
            (void)hipGraphDestroy(captured);
            if (made != hipSuccess) {
                b->edit_graph = nullptr;
                return DINARA_OUT_OF_MEMORY;
            }
        }
        if (hipEventRecord(ctx->start, ctx->stream) != hipSuccess ||
            hipGraphLaunch(b->edit_graph, ctx->stream) != hipSuccess)
            return DINARA_OUT_OF_MEMORY;
        b->graph_used = 1;
    } else {
        if (hipEventRecord(ctx->start, ctx->stream) != hipSuccess) return DINARA_OUT_OF_MEMORY;
        if (const int64_t code = enqueue_unit(b, a, b->timed, trace)) return code;
    }
    if (hipEventRecord(ctx->sweep_stop, ctx->stream) != hipSuccess) return DINARA_OUT_OF_MEMORY;
    // Pairs whose decisions found no room: trace them in further passes, the arena emptied each time.
    int32_t deferred = 0;
    if (trace) {
        if (!b->deferred_count.read(ctx, &deferred, 4)) return DINARA_OUT_OF_MEMORY;
        if (deferred > 0) ctx->arena_wanted = 2 * b->arena_capacity;
        while (deferred > 0) {
            b->trace_passes += 1;
            if (hipMemcpyAsync(b->deferred_held.ptr, b->deferred.ptr, (size_t)deferred * 4, hipMemcpyDeviceToDevice,
                               ctx->stream) != hipSuccess)
                return DINARA_OUT_OF_MEMORY;
            launch_edit_requeue(a, static_cast<const int32_t *>(b->deferred_held.ptr), deferred, ctx->stream);
            sweep_bins(b, a, true, b->trace_reach, ctx->stream, TRACE_MARKS, false, 0);
            join_bins(b, b->trace_reach, TRACE_MARKS);
            walk_slots(b, a, ctx->stream, ctx->side(SIDE_WIDE), WALK_MARKS + 3, false);
            int32_t left = 0;
            if (hipPeekAtLastError() != hipSuccess || !b->deferred_count.read(ctx, &left, 4)) return DINARA_OUT_OF_MEMORY;
            if (left >= deferred) return DINARA_OUT_OF_MEMORY;  // a pair larger than the whole arena
            deferred = left;
        }
    }
    if (hipEventRecord(ctx->stop, ctx->stream) != hipSuccess || hipEventSynchronize(ctx->stop) != hipSuccess)
        return DINARA_OUT_OF_MEMORY;
    float total = 0, sweeps = 0;
    (void)hipEventElapsedTime(&total, ctx->start, ctx->stop);
    (void)hipEventElapsedTime(&sweeps, ctx->start, ctx->sweep_stop);
    b->run_ms = total;
    b->sweep_ms = sweeps;
    // The device counters (sweeps, word-columns, first bands proven) are read back only when asked for: a
    // short batch's run is then one graph launch and one wait.
    b->stats_pending = true;
    b->stats_slots = slots;
    if (!graph && b->timed) {
        const auto spent = [&](int ev, int bin) {
            float ms = 0;
            const int pair = ev + timing_pair(b, bin);
            return hipEventElapsedTime(&ms, ctx->event(pair), ctx->event(pair + 1)) == hipSuccess ? (double)ms : 0.0;
        };
        const bool traced = trace && !b->keep_first;
        for (int bin = 0; bin < EDIT_BINS; ++bin) {
            if (b->first_count[bin] > 0) b->edit_ms[bin] += spent(EV_FIRST, bin);
            if (b->retry_reach[bin] > 0) b->edit_ms[bin] += spent(EV_RETRY, bin);
            if (traced && b->trace_reach[bin] > 0) b->trace_ms[bin] = spent(EV_TRACE, bin);
        }
    }
    if (!graph && trace && b->timed) {
        float ms = 0;
        (void)hipEventElapsedTime(&ms, ctx->event(EV_WALK), ctx->event(EV_WALK + 1));
        b->walk_ms = ms;
    }
    if (graph) b->launches = 1;
    b->ran = true;
    return 0;
}

// A slot's first strip band: its start and end diagonals', widened to a strip's columns (a strip's rows are the band's
// and its columns', so up to there a band is cheap), inside the matrix.
int4 first_strip_band(const dinara_batch *b, int32_t s) {
    const int n = b->rows[s], m = b->cols[s];
    int lo = b->first_low[s], hi = b->first_high[s];
    const int more = strip_columns(strip_c(m)) - (hi - lo + 1);
    if (more > 0 && !b->free_ends) {
        lo = std::max(lo - more / 2, -n);
        hi = std::min(hi + more / 2, m);
    }
    return make_int4(s, lo, hi, 0);
}

// Where, among the classes' timing events, those of a group class's long pairs are (a strip class's, which has none).
constexpr int LONG_PART = CLASS_STRIP_FIRST + 1;

// Sweeps every slot of the first lists until each is settled or left unsettled: want bands from first_low_d /
// first_high_d, round 0 the first lists, each later round the lists the round before filed, kept on the device,
// two sets taking turns. Only the counts come back to the host, and the pairs filed for strips, which the host plans.
// A round's launches (the strips' and each other class's) run side by side: each lasts as long as its longest pair, and
// one after another the classes of 2,000 uneven pairs took 149 ms. Caller holds the device lock.
int64_t sweep_rounds(dinara_batch *b, size_t &arena_index) {
    DeviceContext *ctx = b->ctx;
    const int64_t slots = (int64_t)b->slot_pair.size();
    if (slots == 0) return 0;
    if (hipMemcpyAsync(b->want_low.ptr, b->first_low_d.ptr, slots * 4, hipMemcpyDeviceToDevice, ctx->stream) !=
            hipSuccess ||
        hipMemcpyAsync(b->want_high.ptr, b->first_high_d.ptr, slots * 4, hipMemcpyDeviceToDevice, ctx->stream) !=
            hipSuccess ||
        hipMemsetAsync(b->status.ptr, 0xFF, slots * 4, ctx->stream) != hipSuccess)
        return DINARA_OUT_OF_MEMORY;
    int64_t counts[CLASSES] = {};
    for (int c = 0; c < CLASS_STRIP_FIRST; ++c) counts[c] = b->first_offset[c + 1] - b->first_offset[c];
    // The strip bands a round plans, and how many there are.
    std::vector<int4> bands;
    size_t strips = (size_t)(b->first_offset[CLASSES] - b->first_offset[CLASS_STRIP_FIRST]);
    const auto list_first_strips = [&]() {
        bands.reserve(strips);
        for (int c = CLASS_STRIP_FIRST; c < CLASSES; ++c)
            for (int32_t s : b->first_lists[c]) bands.push_back(first_strip_band(b, s));
    };
    int32_t *lists = static_cast<int32_t *>(b->retry_lists.ptr);
    int32_t *count_d = static_cast<int32_t *>(b->retry_counts.ptr);
    const size_t capacity = (size_t)std::max<int64_t>(slots, 1);
    const SweepArgs args = sweep_args(b);
    for (int round = 0; round < 64; ++round) {
        int64_t pending = (int64_t)strips;
        for (int c = 0; c < CLASS_STRIP_FIRST; ++c) pending += counts[c];
        if (pending == 0) break;
        SweepArgs a = args;
        a.retry_lists = lists + (size_t)(round % 2) * CLASSES * capacity;
        a.retry_counts = count_d + (round % 2) * CLASSES;
        a.strip_retries = static_cast<int4 *>(b->strip_retries.ptr) + (size_t)(round % 2) * capacity;
        const int32_t *in_lists = lists + (size_t)((round + 1) % 2) * CLASSES * capacity;
        StripParts later;
        const bool first = round == 0 && b->phase <= 1;
        StripParts &of = first ? b->first_strips : later;
        DeviceBuffer &plan = first ? b->first_strip_plan : b->strip_plan;
        if (strips > 0) {
            if (!first || !b->first_strips_planned) {
                if (round == 0) list_first_strips();
                of = plan_strips(b, bands, a.record != 0, true);
                if (!upload_strips(b, plan)) return DINARA_OUT_OF_MEMORY;
                b->first_strips_planned = b->first_strips_planned || first;
            }
            if (!reserve_strips(b, of)) return DINARA_OUT_OF_MEMORY;
        }
        if (hipMemsetAsync(a.retry_counts, 0, CLASSES * 4, ctx->stream) != hipSuccess) return DINARA_OUT_OF_MEMORY;
        (void)hipEventRecord(ctx->sweep_start, ctx->stream);
        // The launches in turn on the main stream and the side streams, the strips first.
        (void)hipEventRecord(ctx->mark(0), ctx->stream);
        int turn = 0;
        bool forked[SWEEP_STREAMS] = {};
        const auto next_stream = [&]() {
            const int k = turn++ % SWEEP_STREAMS;
            if (k == 0) return ctx->stream;
            if (!forked[k]) (void)hipStreamWaitEvent(ctx->side(k - 1), ctx->mark(0), 0);
            forked[k] = true;
            return ctx->side(k - 1);
        };
        bool was_timed[CLASSES] = {};
        const auto timed = [&](int c, auto launch) -> int64_t {
            hipStream_t stream = next_stream();
            was_timed[c] = true;
            (void)hipEventRecord(ctx->event(2 * c), stream);
            if (const int64_t code = launch(stream)) return code;
            (void)hipEventRecord(ctx->event(2 * c + 1), stream);
            return 0;
        };
        if (strips > 0) {
            for (int c = CLASS_STRIP_FIRST; c < CLASSES; ++c) b->class_pairs[c] += of.class_pairs[c];
            b->class_launches[CLASS_STRIP_FIRST] += 1;
            if (const int64_t code = timed(CLASS_STRIP_FIRST, [&](hipStream_t stream) {
                    return launch_strips(b, a, of, plan, false, stream);
                }))
                return code;
        }
        for (int c = CLASS_STRIP_FIRST - 1; c >= 0; --c) {
            if (counts[c] == 0) continue;
            const int32_t *list = round == 0 ? static_cast<const int32_t *>(b->first_lists_d.ptr) + b->first_offset[c]
                                             : in_lists + (size_t)c * capacity;
            // The narrow group bands' long pairs (the first of their list, longest side first) in a launch of their own
            // where the list would not all run at once with the LDS they take: the letters a launch stages are its
            // longest pair's.
            int64_t longs = 0;
            if (c <= CLASS_GROUP64 && round == 0 && b->limits.group_narrow > b->limits.group_letters) {
                for (int64_t i = 0; i < counts[c]; ++i) {
                    const int32_t s = b->first_lists[c][i];
                    if (b->rows[s] + b->cols[s] > b->limits.group_letters) longs = i + 1;
                }
                const int64_t at_once = LDS_BYTES / (4 * group_region(b->limits.group_narrow)) * ctx->compute_units;
                if (longs > 0 && (counts[c] + 3) / 4 <= at_once) longs = counts[c];
            }
            const int longest = band_is_wave(c) ? (b->user_band              ? b->max_letters
                                                   : c == CLASS_WAVE_FIRST ? b->limits.wave_letters
                                                                           : b->limits.wave128_letters)
                                : c <= CLASS_GROUP64 && longs == 0 && round == 0 ? b->limits.group_letters
                                                                                 : group_limit(b->limits, c);
            if (longs > 0)
                if (const int64_t code = timed(LONG_PART + c, [&](hipStream_t stream) {
                        return launch_class(b, a, c, list, longs, longest, arena_index, stream);
                    }))
                    return code;
            if (counts[c] > longs)
                if (const int64_t code = timed(c, [&](hipStream_t stream) {
                        return launch_class(b, a, c, list + longs, counts[c] - longs,
                                            longs > 0 ? b->limits.group_letters : longest, arena_index, stream);
                    }))
                    return code;
        }
        for (int k = 1; k < SWEEP_STREAMS; ++k) {
            if (!forked[k]) continue;
            (void)hipEventRecord(ctx->mark(k), ctx->side(k - 1));
            (void)hipStreamWaitEvent(ctx->stream, ctx->mark(k), 0);
        }
        (void)hipEventRecord(ctx->sweep_stop, ctx->stream);
        int32_t filed[CLASSES];
        if (hipMemcpyAsync(filed, a.retry_counts, sizeof(filed), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
            hipStreamSynchronize(ctx->stream) != hipSuccess)
            return DINARA_OUT_OF_MEMORY;
        float ms = 0;
        (void)hipEventElapsedTime(&ms, ctx->sweep_start, ctx->sweep_stop);
        b->sweep_ms += ms;
        int64_t retried = 0;
        for (int c = 0; c <= LONG_PART + CLASS_GROUP64; ++c) {
            if (!was_timed[c]) continue;
            float class_ms = 0;
            (void)hipEventElapsedTime(&class_ms, ctx->event(2 * c), ctx->event(2 * c + 1));
            b->class_ms[c < LONG_PART ? c : c - LONG_PART] += class_ms;
        }
        for (int c = 0; c <= CLASS_STRIP_FIRST; ++c) {
            counts[c] = filed[c];
            retried += filed[c];
        }
        b->expired = b->expired || filed[STRIP_EXPIRED] > 0;
        strips = (size_t)filed[CLASS_STRIP_FIRST];
        bands.resize(strips);
        if (strips > 0) {
            if (hipMemcpyAsync(bands.data(), a.strip_retries, strips * sizeof(int4), hipMemcpyDeviceToHost, ctx->stream) !=
                    hipSuccess ||
                hipStreamSynchronize(ctx->stream) != hipSuccess)
                return DINARA_OUT_OF_MEMORY;
            // Longest first (slots are): the launch's longest pipelines claim their strips first.
            std::sort(bands.begin(), bands.end(), [](const int4 &x, const int4 &y) { return x.x < y.x; });
        }
        if (round == 0 && b->phase <= 1) b->first_proven = (double)(slots - retried);
    }
    return 0;
}

// The forward phase's views, free letters, bands and lists onto the device. Caller holds the device lock.
int64_t free_phase_a(dinara_batch *b) {
    DeviceContext *ctx = b->ctx;
    const size_t slots = b->slot_pair.size();
    if (slots == 0) return 0;
    b->phase = 1;
    b->first_offset = b->a_first_offset;
    b->first_low = b->a_first_low;
    b->first_high = b->a_first_high;
    for (int c = 0; c < CLASSES; ++c)
        b->first_lists[c].assign(b->a_first_all.begin() + b->a_first_offset[c],
                                 b->a_first_all.begin() + b->a_first_offset[c + 1]);
    if (!b->view_rows_d.write(ctx, b->a_rows.data(), slots * 4) || !b->view_cols_d.write(ctx, b->a_cols.data(), slots * 4) ||
        !b->view_ref_at_d.write(ctx, b->a_at.data(), slots * 4) || !b->view_qry_at_d.write(ctx, b->a_at.data(), slots * 4) ||
        !b->free_d.write(ctx, b->a_free.data(), slots * 16) ||
        !b->first_low_d.write(ctx, b->a_first_low.data(), slots * 4) ||
        !b->first_high_d.write(ctx, b->a_first_high.data(), slots * 4) ||
        !b->first_lists_d.upload(ctx, b->a_first_all.data(), b->a_first_all.size() * 4))
        return DINARA_OUT_OF_MEMORY;
    return 0;
}

// The anchored phase of free-end alignments, from the forward phase's results: each settled pair (within the cap)
// sweeps the letters before its end, back from the end (no free start), free to end where the forward phase was
// free to start, its band the one its known cost proves; a pair it settles is walked from the end it finds.
// Caller holds the device lock.
int64_t free_phase_b(dinara_batch *b) {
    DeviceContext *ctx = b->ctx;
    const int64_t slots = (int64_t)b->slot_pair.size();
    b->a_status_h.resize(slots);
    b->a_cost_h.resize(slots);
    b->a_end_row_h.resize(slots);
    b->a_end_col_h.resize(slots);
    if (!b->status.read(ctx, b->a_status_h.data(), slots * 4) || !b->cost.read(ctx, b->a_cost_h.data(), slots * 4) ||
        !b->end_row_d.read(ctx, b->a_end_row_h.data(), slots * 4) ||
        !b->end_col_d.read(ctx, b->a_end_col_h.data(), slots * 4))
        return DINARA_OUT_OF_MEMORY;
    const CostParams &c = b->costs;
    auto gap = [&](int64_t k, int open, int ext, int open2, int ext2) -> int64_t {
        if (k <= 0) return 0;
        const int64_t one = (int64_t)open + k * ext;
        return c.pieces == 2 ? std::min(one, (int64_t)open2 + k * ext2) : one;
    };
    const bool right = b->options.right_ties;
    const int64_t cap = b->options.max_cost >= 0 ? b->options.max_cost : INT64_MAX / 4;
    std::vector<int32_t> rows(slots), cols(slots), ref_at(slots), qry_at(slots), fr((size_t)slots * 4, 0);
    b->b_rows_h.assign(slots, 0);
    b->b_cols_h.assign(slots, 0);
    for (auto &l : b->first_lists) l.clear();
    for (int64_t s = 0; s < slots; ++s) {
        const int32_t n = b->rows[s], m = b->cols[s];
        const int32_t re = b->a_end_row_h[s], ce = b->a_end_col_h[s];
        const bool go = b->a_status_h[s] == 0 && b->a_cost_h[s] <= cap;
        rows[s] = go ? re : 0;
        cols[s] = go ? ce : 0;
        ref_at[s] = go && right ? n - re : 0;
        qry_at[s] = go && right ? m - ce : 0;
        b->b_rows_h[s] = rows[s];
        b->b_cols_h[s] = cols[s];
        if (!go) continue;
        // Free to end where the forward phase was free to start.
        const int32_t er = std::min<int32_t>(b->a_free[4 * s], re), ec = std::min<int32_t>(b->a_free[4 * s + 2], ce);
        fr[4 * s + 1] = er;
        fr[4 * s + 3] = ec;
        const int64_t least = b->a_cost_h[s], target = least + 1, end = (int64_t)ce - re;
        auto off = [&](int64_t k) -> int64_t {  // off_band_ends with no free start
            const int64_t high = std::max<int64_t>(0, end + er), low = std::min<int64_t>(0, end - ec);
            if (k > high) return gap(k, c.ins_open, c.ins_ext, c.ins_open2, c.ins_ext2) +
                                 gap(k - (end + er), c.del_open, c.del_ext, c.del_open2, c.del_ext2);
            if (k < low) return gap(-k, c.del_open, c.del_ext, c.del_open2, c.del_ext2) +
                                gap(end - ec - k, c.ins_open, c.ins_ext, c.ins_open2, c.ins_ext2);
            return 0;
        };
        int64_t h = std::max<int64_t>(0, end + er), l = std::min<int64_t>(0, end - ec);
        while (h < ce && off(h + 1) < target) ++h;
        while (l > -re && off(l - 1) < target) --l;
        b->first_low[s] = (int32_t)l;
        b->first_high[s] = (int32_t)h;
        const int cls = first_class(b, s, (int)(h - l + 1));
        if (cls != CLASS_TOO_WIDE) b->first_lists[cls].push_back((int32_t)s);
    }
    std::vector<int32_t> first_all;
    b->first_offset.assign(CLASSES + 1, 0);
    for (int k = 0; k < CLASSES; ++k) {
        b->first_offset[k] = (int64_t)first_all.size();
        first_all.insert(first_all.end(), b->first_lists[k].begin(), b->first_lists[k].end());
    }
    b->first_offset[CLASSES] = (int64_t)first_all.size();
    if (first_all.empty()) first_all.push_back(0);
    if (!b->view_rows_d.write(ctx, rows.data(), slots * 4) || !b->view_cols_d.write(ctx, cols.data(), slots * 4) ||
        !b->view_ref_at_d.write(ctx, ref_at.data(), slots * 4) || !b->view_qry_at_d.write(ctx, qry_at.data(), slots * 4) ||
        !b->free_d.write(ctx, fr.data(), slots * 16) || !b->first_low_d.write(ctx, b->first_low.data(), slots * 4) ||
        !b->first_high_d.write(ctx, b->first_high.data(), slots * 4) ||
        !b->first_lists_d.upload(ctx, first_all.data(), first_all.size() * 4))
        return DINARA_OUT_OF_MEMORY;
    b->phase = 2;
    return 0;
}

// The decision bytes one pair may take on the whole-matrix path: past it the pair stays unsettled.
constexpr size_t FULL_BUDGET = size_t(16) << 30;

// After a run, every pair the band sweeps left unsettled (wider than the widest band, more letters than the strips
// take in bands, or left by a strip's expired wait) is swept whole and walked (strip.hip); a pair under free
// ends or a user band, or whose decisions pass FULL_BUDGET, stays unsettled. A batch none of
// whose pairs could need it skips the pass; otherwise the unsettled slots are listed on the device and only their
// count (and list) come back. Caller holds the device lock.
int64_t full_pass(dinara_batch *b) {
    DeviceContext *ctx = b->ctx;
    const int64_t slots = (int64_t)b->slot_pair.size();
    b->full_pairs = b->full_ms = 0;
    if (b->free_ends || b->user_band || slots == 0) return 0;
    if (b->may_need_full < 0) {
        // Under both the unit bins and the band classes a band of 8192 diagonals proves any pair of fewer letters,
        // and such a pair fits every kernel's LDS.
        b->may_need_full = 0;
        for (int64_t s = 0; s < slots; ++s)
            if ((int64_t)b->rows[s] + b->cols[s] + 3 > 8192) b->may_need_full = 1;
    }
    if (!b->may_need_full && !b->whole && !b->expired) return 0;
    const auto began = std::chrono::steady_clock::now();
    if (!b->full_list.reserve((size_t)slots * 4) || !b->full_count.reserve(4) ||
        hipMemsetAsync(b->full_count.ptr, 0, 4, ctx->stream) != hipSuccess)
        return DINARA_OUT_OF_MEMORY;
    launch_collect_unsettled(static_cast<const int32_t *>(b->status.ptr), (int)slots,
                             static_cast<int32_t *>(b->full_list.ptr), static_cast<int32_t *>(b->full_count.ptr),
                             ctx->stream);
    int32_t count = 0;
    if (hipPeekAtLastError() != hipSuccess || !b->full_count.read(ctx, &count, 4)) return DINARA_OUT_OF_MEMORY;
    if (count == 0) return 0;
    std::vector<int32_t> list(count);
    if (!b->full_list.read(ctx, list.data(), (size_t)count * 4)) return DINARA_OUT_OF_MEMORY;
    std::sort(list.begin(), list.end());
    const bool record = b->kind == DINARA_BATCH_ALIGNMENTS;
    const size_t record_bytes = b->costs.pieces == 2 ? 8 : 4;
    std::vector<int4> bands;
    for (const int32_t slot : list) {
        if (slot < 0 || slot >= slots) continue;
        const int64_t n = b->rows[slot], m = b->cols[slot];
        const int64_t strips = std::max<int64_t>(1, (m + strip_columns(8) - 1) / strip_columns(8));
        if (record && (size_t)(strips * n * 64) * record_bytes > FULL_BUDGET) continue;
        bands.push_back(make_int4(slot, (int)-n, (int)m, 0));
    }
    if (!bands.empty()) {
        const StripParts of = plan_strips(b, bands, record, false);
        if (!upload_strips(b, b->strip_plan) || !reserve_strips(b, of)) return DINARA_OUT_OF_MEMORY;
        if (const int64_t code = launch_strips(b, sweep_args(b), of, b->strip_plan, true, ctx->stream)) return code;
    }
    b->full_pairs = (double)bands.size();
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return DINARA_OUT_OF_MEMORY;
    b->full_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - began).count();
    return 0;
}

int64_t run(dinara_batch *b) {
    DeviceContext *ctx = b->ctx;
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    (void)hipGetLastError();  // an earlier, unrelated call's error is not this run's
    if (b->whole) {
        // No band sweep: every slot unsettled, then the whole-matrix pass takes them all.
        const int64_t slots = (int64_t)b->slot_pair.size();
        b->launches = b->first_proven = 0;
        b->run_ms = b->sweep_ms = b->walk_ms = 0;
        if (slots > 0 && (hipMemsetAsync(b->status.ptr, 0xFF, slots * 4, ctx->stream) != hipSuccess ||
                          (b->kind == DINARA_BATCH_ALIGNMENTS &&
                           hipMemsetAsync(b->cigar_used.ptr, 0, 8, ctx->stream) != hipSuccess)))
            return DINARA_OUT_OF_MEMORY;
        const int64_t code = full_pass(b);
        b->run_ms = b->full_ms;
        b->ran = code == 0;
        return code;
    }
    if (b->unit) {
        if (const int64_t code = run_unit(b, true)) return code;
        return full_pass(b);
    }
    const int64_t slots = (int64_t)b->slot_pair.size();
    b->launches = b->first_proven = 0;
    b->expired = false;
    b->run_ms = b->sweep_ms = b->walk_ms = 0;
    for (int c = 0; c < CLASSES; ++c) b->class_ms[c] = b->class_launches[c] = b->class_pairs[c] = 0;
    if (hipEventRecord(ctx->start, ctx->stream) != hipSuccess) return DINARA_OUT_OF_MEMORY;
    if (slots > 0 && b->kind == DINARA_BATCH_ALIGNMENTS &&
        hipMemsetAsync(b->cigar_used.ptr, 0, 8, ctx->stream) != hipSuccess)
        return DINARA_OUT_OF_MEMORY;
    size_t arena_index = 0;
    if (b->free_ends) {
        // Free ends: the forward phase finds each pair's cost and end (reference tests/test_alignment.mojo:1983-2000);
        // alignments sweep again from that end, anchored, keeping decisions, for the start and the walk.
        if (const int64_t code = free_phase_a(b)) return code;
        b->phase = 1;
        if (const int64_t code = sweep_rounds(b, arena_index)) return code;
        if (b->kind == DINARA_BATCH_ALIGNMENTS && slots > 0) {
            if (const int64_t code = free_phase_b(b)) return code;
            b->phase = 2;
            if (const int64_t code = sweep_rounds(b, arena_index)) return code;
        }
    } else if (const int64_t code = sweep_rounds(b, arena_index)) {
        return code;
    }
    if (b->kind == DINARA_BATCH_ALIGNMENTS && slots > 0) {
        SweepArgs a = sweep_args(b);
        (void)hipEventRecord(ctx->event(2 * CLASSES), ctx->stream);
        launch_walk(a, ctx->stream);
        (void)hipEventRecord(ctx->event(2 * CLASSES + 1), ctx->stream);
    }
    if (hipEventRecord(ctx->stop, ctx->stream) != hipSuccess || hipEventSynchronize(ctx->stop) != hipSuccess)
        return DINARA_OUT_OF_MEMORY;
    if (b->kind == DINARA_BATCH_ALIGNMENTS && slots > 0) {
        float walk_ms = 0;
        (void)hipEventElapsedTime(&walk_ms, ctx->event(2 * CLASSES), ctx->event(2 * CLASSES + 1));
        b->walk_ms = walk_ms;
    }
    float total = 0;
    (void)hipEventElapsedTime(&total, ctx->start, ctx->stop);
    b->run_ms = total;
    b->ran = true;
    return full_pass(b);
}

// A small batch's results in one copy: everything of the region from the first of them to the last (up to 1 MiB, most
// of it the CIGARs' room), rather than six copies waited for one after another.
constexpr int64_t SMALL_FETCH = 256;

int64_t fetch_at_once(dinara_batch *b) {
    const int64_t slots = (int64_t)b->slot_pair.size();
    const bool aligned = b->kind == DINARA_BATCH_ALIGNMENTS, ends = aligned && b->free_ends;
    DeviceBuffer *wanted[] = {&b->cost, &b->status, ends ? &b->end_row_d : nullptr, ends ? &b->end_col_d : nullptr,
                              aligned ? &b->cigar_used : nullptr, aligned ? &b->cigar_offset : nullptr,
                              aligned ? &b->cigar_length : nullptr, aligned ? &b->cigars : nullptr};
    const uint8_t *base = b->region.base;
    const uint8_t *first = base + b->region.size, *last = base;
    for (DeviceBuffer *buffer : wanted)
        if (buffer && b->region.holds(buffer->ptr, buffer->size)) {
            const uint8_t *at = static_cast<const uint8_t *>(buffer->ptr);
            first = std::min(first, at);
            last = std::max(last, at + buffer->size);
        }
    if (last > first && (hipMemcpyAsync(b->region.image + (first - base), first, last - first, hipMemcpyDeviceToHost,
                                        b->ctx->stream) != hipSuccess ||
                         hipStreamSynchronize(b->ctx->stream) != hipSuccess))
        return DINARA_OUT_OF_MEMORY;
    auto read = [&](DeviceBuffer &buffer, void *host, size_t bytes) {
        if (bytes > buffer.size) return false;
        if (!b->region.holds(buffer.ptr, buffer.size)) return buffer.read(b->ctx, host, bytes);
        std::memcpy(host, b->region.image + (static_cast<uint8_t *>(buffer.ptr) - base), bytes);
        return true;
    };
    if (!read(b->cost, b->cost_h.data(), slots * 4) || !read(b->status, b->status_h.data(), slots * 4))
        return DINARA_OUT_OF_MEMORY;
    if (ends) {
        b->b_end_row_h.resize(slots);
        b->b_end_col_h.resize(slots);
        if (!read(b->end_row_d, b->b_end_row_h.data(), slots * 4) ||
            !read(b->end_col_d, b->b_end_col_h.data(), slots * 4))
            return DINARA_OUT_OF_MEMORY;
    }
    if (aligned) {
        unsigned long long used = 0;
        b->cigar_offset_h.resize(slots);
        b->cigar_length_h.resize(slots);
        if (!read(b->cigar_used, &used, 8) || !read(b->cigar_offset, b->cigar_offset_h.data(), slots * 8) ||
            !read(b->cigar_length, b->cigar_length_h.data(), slots * 4))
            return DINARA_OUT_OF_MEMORY;
        b->cigars_h.resize(std::max<unsigned long long>(used, 1));
        if (used > 0 && !read(b->cigars, b->cigars_h.data(), used)) return DINARA_OUT_OF_MEMORY;
    }
    return 0;
}

int64_t fetch(dinara_batch *b) {
    DeviceContext *ctx = b->ctx;
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    const int64_t slots = (int64_t)b->slot_pair.size();
    b->cost_h.resize(slots);
    b->status_h.resize(slots);
    if (slots == 0) return 0;
    if (b->region.image && slots <= SMALL_FETCH) return fetch_at_once(b);
    if (!b->cost.read(ctx, b->cost_h.data(), slots * 4) || !b->status.read(ctx, b->status_h.data(), slots * 4))
        return DINARA_OUT_OF_MEMORY;
    if (b->free_ends && b->kind == DINARA_BATCH_ALIGNMENTS) {
        b->b_end_row_h.resize(slots);
        b->b_end_col_h.resize(slots);
        if (!b->end_row_d.read(ctx, b->b_end_row_h.data(), slots * 4) ||
            !b->end_col_d.read(ctx, b->b_end_col_h.data(), slots * 4))
            return DINARA_OUT_OF_MEMORY;
    }
    if (b->kind == DINARA_BATCH_ALIGNMENTS) {
        unsigned long long used = 0;
        b->cigar_offset_h.resize(slots);
        b->cigar_length_h.resize(slots);
        if (!b->cigar_used.read(ctx, &used, 8) || !b->cigar_offset.read(ctx, b->cigar_offset_h.data(), slots * 8) ||
            !b->cigar_length.read(ctx, b->cigar_length_h.data(), slots * 4))
            return DINARA_OUT_OF_MEMORY;
        b->cigars_h.resize(std::max<unsigned long long>(used, 1));
        if (used > 0 && !b->cigars.read(ctx, b->cigars_h.data(), used)) return DINARA_OUT_OF_MEMORY;
    }
    return 0;
}

// A pair's code when the device left it unsettled (a nonzero status): no result.
int64_t unsettled_code(int32_t) { return DINARA_OUT_OF_MEMORY; }

dinara_batch *batch_new(int64_t gpu, int64_t kind, int64_t pairs, const char *const *refs, const int64_t *ref_lens,
                        const char *const *qrys, const int64_t *qry_lens, const dinara_costs *costs,
                        const dinara_mode *mode, const dinara_options *options, int64_t threads, int64_t *status) {
    auto fail = [&](int64_t code) -> dinara_batch * {
        if (status) *status = code;
        return nullptr;
    };
    ParsedCosts parsed = parse_costs(costs);
    if (parsed.code) return fail(parsed.code);
    if (const int64_t code = check_mode(mode)) return fail(code);
    if (kind != DINARA_BATCH_DISTANCES && kind != DINARA_BATCH_ALIGNMENTS) return fail(DINARA_INVALID_MODE);
    DeviceContext *ctx = device_context(gpu);
    if (!ctx) return fail(DINARA_NO_DEVICE);
    auto *b = new dinara_batch();
    b->gpu = (int)gpu;
    b->ctx = ctx;
    b->kind = kind;
    b->pairs = std::max<int64_t>(pairs, 0);
    // Packing threads: as many as asked, but no more than one a half-million letters (a thread's start costs more
    // than packing fewer letters).
    {
        int64_t letters = 0;
        for (int64_t i = 0; i < b->pairs; ++i)
            letters += std::max<int64_t>(ref_lens[i], 0) + std::max<int64_t>(qry_lens[i], 0);
        threads = std::max<int64_t>(1, std::min<int64_t>(threads, letters >> 19));
    }
    b->threads = threads;
    b->parsed = parsed;
    b->options = parse_options(options);
    b->lds_limit = ctx->lds_limit;
    if (const char *w = std::getenv("DINARA_INITIAL_WIDTH")) b->initial_width = std::max(1, atoi(w));
    CostParams &c = b->costs;
    c.mismatch = (int)parsed.mismatch;
    c.del_open = (int)parsed.del_opening;
    c.del_ext = (int)parsed.del_extension;
    c.ins_open = (int)parsed.opening;
    c.ins_ext = (int)parsed.extension;
    c.del_first = c.del_open + c.del_ext;
    c.ins_first = c.ins_open + c.ins_ext;
    c.pieces = parsed.two_piece ? 2 : 1;
    c.del_open2 = (int)parsed.del_opening2;
    c.del_ext2 = (int)parsed.del_extension2;
    c.ins_open2 = (int)parsed.opening2;
    c.ins_ext2 = (int)parsed.extension2;
    c.del_first2 = c.del_open2 + c.del_ext2;
    c.ins_first2 = c.ins_open2 + c.ins_ext2;
    // The lanes' diagonals are the query's letters less the reference's: the library band mirrored
    // (lanes.mojo:1151-1155).
    const Options &o = b->options;
    b->user_band = o.band_low > -UNBOUNDED || o.band_high < UNBOUNDED;
    const int64_t clamp = int64_t(1) << 30;
    b->user_low = (int)std::max<int64_t>(-o.band_high, -clamp);
    b->user_high = (int)std::min<int64_t>(-o.band_low, clamp);
    // Unit costs times a scale, with no user band, take the bit-parallel path (DINARA_GOTOH_UNIT=1 keeps them on the
    // gap-cost sweeps, for comparison).
    b->free_ends = free_mode(mode);
    if (b->free_ends) {
        // Free ends under a user band are not served (the band would move with every view).
        if (b->user_band) {
            delete b;
            return fail(DINARA_INVALID_MODE);
        }
        b->ends[0] = mode->reference_start;
        b->ends[1] = mode->reference_end;
        b->ends[2] = mode->query_start;
        b->ends[3] = mode->query_end;
    }
    b->unit = !b->user_band && !b->free_ends && !parsed.two_piece && parsed.opening == 0 && parsed.del_opening == 0 &&
              parsed.extension == parsed.mismatch && parsed.del_extension == parsed.mismatch &&
              !(std::getenv("DINARA_GOTOH_UNIT") && std::atoi(std::getenv("DINARA_GOTOH_UNIT")) != 0);
    b->unit_scale = (int)parsed.mismatch;
    int64_t dearest = std::max<int64_t>(
        parsed.mismatch, std::max(parsed.opening + parsed.extension, parsed.del_opening + parsed.del_extension));
    if (parsed.two_piece)
        dearest = std::max(dearest, std::max(parsed.opening2 + parsed.extension2, parsed.del_opening2 + parsed.del_extension2));
    b->dearest = std::max<int64_t>(dearest, 1);
    b->code.assign(b->pairs, 0);
    b->plain.assign(b->pairs, 0);
    b->reference_length.assign(b->pairs, 0);
    b->query_length.assign(b->pairs, 0);
    const bool capped = o.max_cost >= 0;
    parallel_for(b->pairs, threads, [&](int64_t lo, int64_t hi) {
        for (int64_t i = lo; i < hi; ++i) {
            const int64_t n = ref_lens[i], m = qry_lens[i];
            b->plain[i] = n >= 0 && m >= 0 && Dna::plain(refs[i], n) && Dna::plain(qrys[i], m);
            int64_t code = b->plain[i] ? 0 : pair_code(refs[i], n, qrys[i], m);
            if (code == 0) {
                // Every cost the sweep holds stays well inside 32 bits.
                if ((n + m + 4) * dearest >= REAL_LIMIT || n >= (int64_t(1) << 28) || m >= (int64_t(1) << 28))
                    code = DINARA_OUT_OF_MEMORY;
            }
            if (code == 0 && b->user_band) {
                // No alignment inside a band missing the start's or the end's diagonal (lanes.mojo:1363-1367).
                const int64_t end = m - n;
                if (b->user_low > 0 || b->user_high < 0 || b->user_low > end || b->user_high < end)
                    code = capped ? DINARA_ABOVE_MAX : DINARA_OUTSIDE_BAND;
            }
            b->code[i] = code;
            b->reference_length[i] = std::max<int64_t>(n, 0);
            b->query_length[i] = std::max<int64_t>(m, 0);
        }
    });
    int64_t code;
    {
        std::lock_guard<std::mutex> serial(ctx->lock);
        DeviceGuard guard(ctx);
        code = prepare(b, refs, qrys);
    }
    if (code) {
        delete b;
        return fail(code);
    }
    if (status) *status = 0;
    return b;
}

}  // namespace

// ------------------------------------------------------------------ the C ABI

extern "C" {

void dinara_free(char *cigar) { std::free(cigar); }

int64_t dinara_device_count(void) { return device_count(); }

dinara_batch *dinara_batch_new(int64_t gpu, int64_t kind, int64_t pairs, const char *const *references,
                               const int64_t *reference_lengths, const char *const *queries,
                               const int64_t *query_lengths, const dinara_costs *costs, const dinara_mode *mode,
                               const dinara_options *options, int64_t threads, int64_t *status) {
    return batch_new(gpu, kind, pairs, references, reference_lengths, queries, query_lengths, costs, mode, options,
                     threads, status);
}

int64_t dinara_batch_run(dinara_batch *batch) {
    if (!batch) return DINARA_INVALID_MODE;
    return run(batch);
}

int64_t dinara_batch_distances(dinara_batch *b, int64_t *results) {
    if (!b || b->kind != DINARA_BATCH_DISTANCES || !b->ran) return DINARA_INVALID_MODE;
    if (const int64_t code = fetch(b)) return code;
    const bool capped = b->options.max_cost >= 0;
    for (int64_t i = 0; i < b->pairs; ++i) results[i] = b->code[i];
    for (size_t s = 0; s < b->slot_pair.size(); ++s) {
        const int32_t p = b->slot_pair[s];
        if (b->status_h[s] != 0) {
            results[p] = unsettled_code(b->status_h[s]);
            continue;
        }
        const int64_t cost = b->cost_h[s];
        results[p] = capped && cost > b->options.max_cost ? DINARA_ABOVE_MAX : cost;
    }
    return 0;
}

int64_t dinara_batch_alignments(dinara_batch *b, dinara_alignment *alignments, int64_t *statuses) {
    if (!b || b->kind != DINARA_BATCH_ALIGNMENTS || !b->ran) return DINARA_INVALID_MODE;
    if (const int64_t code = fetch(b)) return code;
    const bool capped = b->options.max_cost >= 0;
    for (int64_t i = 0; i < b->pairs; ++i) {
        statuses[i] = b->code[i];
        if (b->code[i] != 0) {
            alignments[i].cigar = nullptr;
            alignments[i].cigar_length = 0;
        }
    }
    std::atomic<bool> oom{false};
    parallel_for((int64_t)b->slot_pair.size(), b->threads, [&](int64_t lo, int64_t hi) {
        for (int64_t s = lo; s < hi; ++s) {
            const int32_t p = b->slot_pair[s];
            dinara_alignment &out = alignments[p];
            out.cigar = nullptr;
            out.cigar_length = 0;
            // Free ends: the cost is the forward phase's, the CIGAR the anchored phase's.
            const int32_t status = b->free_ends ? b->a_status_h[s] : b->status_h[s];
            if (status != 0) {
                statuses[p] = unsettled_code(status);
                continue;
            }
            const int64_t cost = b->free_ends ? b->a_cost_h[s] : b->cost_h[s];
            if (capped && cost > b->options.max_cost) {
                statuses[p] = DINARA_ABOVE_MAX;
                continue;
            }
            if (b->free_ends && b->status_h[s] != 0) {
                statuses[p] = unsettled_code(b->status_h[s]);
                continue;
            }
            const int64_t length = b->cigar_length_h[s];
            char *text = static_cast<char *>(std::malloc(length + 1));
            if (!text) {
                statuses[p] = DINARA_OUT_OF_MEMORY;
                oom.store(true);
                continue;
            }
            std::memcpy(text, b->cigars_h.data() + b->cigar_offset_h[s], length);
            text[length] = 0;
            out.cost = cost;
            out.score = -cost;
            out.reference_start = 0;
            out.reference_end = b->reference_length[p];
            out.query_start = 0;
            out.query_end = b->query_length[p];
            if (b->free_ends) {
                // The forward phase's end and the anchored phase's, as spans of the pair (Ties.RIGHT's mirrored).
                const int64_t n = b->rows[s], m = b->cols[s];
                const int64_t re = b->a_end_row_h[s], ce = b->a_end_col_h[s];
                const int64_t rb = b->b_end_row_h[s], cb = b->b_end_col_h[s];
                if (b->options.right_ties) {
                    out.reference_start = n - re;
                    out.reference_end = n - re + rb;
                    out.query_start = m - ce;
                    out.query_end = m - ce + cb;
                } else {
                    out.reference_start = re - rb;
                    out.reference_end = re;
                    out.query_start = ce - cb;
                    out.query_end = ce;
                }
            }
            out.cigar = text;
            out.cigar_length = length;
            statuses[p] = 0;
        }
    });
    return 0;
}

int64_t dinara_batch_features(dinara_batch *b, float *features) {
    if (!b) return DINARA_INVALID_MODE;
    const int64_t slots = (int64_t)b->slot_pair.size();
    std::fill(features, features + b->pairs * FEATURE_STRIDE, 0.0f);
    if (slots == 0) return 0;
    DeviceContext *ctx = b->ctx;
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    DeviceBuffer out;
    if (!out.reserve((size_t)slots * FEATURE_STRIDE * 4)) return DINARA_OUT_OF_MEMORY;
    SweepArgs a = sweep_args(b);
    launch_features(a.tape, (int)slots, b->reversed ? 1 : 0, static_cast<float *>(out.ptr), ctx->stream);
    std::vector<float> host((size_t)slots * FEATURE_STRIDE);
    if (hipGetLastError() != hipSuccess || !out.read(ctx, host.data(), host.size() * 4)) return DINARA_OUT_OF_MEMORY;
    for (int64_t s = 0; s < slots; ++s)
        std::memcpy(features + (int64_t)b->slot_pair[s] * FEATURE_STRIDE, host.data() + s * FEATURE_STRIDE,
                    FEATURE_STRIDE * 4);
    return 0;
}

}  // extern "C"

namespace {

// Every slot's first band from its guessed cost (`guess_of(slot)`, below zero: no guess), classes and device lists.
template <typename GuessOf>
int64_t seed_slots(dinara_batch *b, GuessOf guess_of) {
    const int64_t slots = (int64_t)b->slot_pair.size();
    if (slots == 0) return 0;
    // The lanes' off-band price (lanes.mojo:333-345) in the batch's costs, as the device's off_band.
    const CostParams &c = b->costs;
    auto ins = [&](int64_t k) {
        if (k <= 0) return int64_t(0);
        const int64_t one = (int64_t)c.ins_open + k * (int64_t)c.ins_ext;
        return c.pieces == 2 ? std::min(one, (int64_t)c.ins_open2 + k * (int64_t)c.ins_ext2) : one;
    };
    auto del = [&](int64_t k) {
        if (k <= 0) return int64_t(0);
        const int64_t one = (int64_t)c.del_open + k * (int64_t)c.del_ext;
        return c.pieces == 2 ? std::min(one, (int64_t)c.del_open2 + k * (int64_t)c.del_ext2) : one;
    };
    auto off = [&](int64_t k, int64_t end) {
        if (k > std::max<int64_t>(end, 0)) return ins(k) + del(k - end);
        if (k < std::min<int64_t>(end, 0)) return del(-k) + ins(end - k);
        return int64_t(0);
    };
    for (auto &l : b->first_lists) l.clear();
    for (int64_t s = 0; s < slots; ++s) {
        const int32_t n = b->rows[s], m = b->cols[s], end = m - n;
        const int64_t guess = guess_of(s);
        int32_t lo = std::min(0, end) - 1, hi = std::max(0, end) + 1;
        if (guess >= 0 && !b->user_band) {
            // The narrowest band whose every outside path costs more than the guess: a pair costing no more than
            // its guess is proven by it at once.
            auto widen = [&](int32_t from, int32_t step, int32_t limit) {
                int32_t k = from, span = 1;
                while (span < (1 << 22) && k + step * span >= -limit - 1 && k + step * span <= limit + 1 &&
                       off(k + step * span, end) <= guess)
                    span *= 2;
                for (; span > 0; span /= 2)
                    if (off(k + step * span, end) <= guess) k += step * span;
                return k;
            };
            hi = std::min(std::max(hi, widen(std::max(0, end), 1, m) + 1), m + 1);
            lo = std::max(std::min(lo, widen(std::min(0, end), -1, n) - 1), -n - 1);
        }
        b->first_low[s] = lo;
        b->first_high[s] = hi;
        const int cls = first_class(b, s, std::max(hi - lo + 1, 32));
        if (cls != CLASS_TOO_WIDE) b->first_lists[cls].push_back((int32_t)s);
    }
    std::vector<int32_t> first_all;
    b->first_offset.assign(CLASSES + 1, 0);
    for (int c2 = 0; c2 < CLASSES; ++c2) {
        b->first_offset[c2] = (int64_t)first_all.size();
        first_all.insert(first_all.end(), b->first_lists[c2].begin(), b->first_lists[c2].end());
    }
    b->first_offset[CLASSES] = (int64_t)first_all.size();
    b->first_strips_planned = false;
    if (first_all.empty()) first_all.push_back(0);  // every pair too wide: the device list still needs room
    DeviceContext *ctx = b->ctx;
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    if (!b->first_low_d.write(ctx, b->first_low.data(), slots * 4) ||
        !b->first_high_d.write(ctx, b->first_high.data(), slots * 4) ||
        !b->first_lists_d.upload(ctx, first_all.data(), std::max<size_t>(first_all.size(), 1) * 4))
        return DINARA_OUT_OF_MEMORY;
    if (b->unit) return unit_lists(b);
    return 0;
}

// The launch shape when the device files each pair's first band: a first queue may hold any pair whose class starts
// at or below the bin and whose widest band reaches it. Caller holds the device lock.
void seeded_shape(dinara_batch *b) {
    bool same = true;
    for (int c = 0; c < EDIT_LENGTH_CLASSES; ++c) same = same && b->seeded_start[c] == b->start_bin[c];
    if (same) return;
    int64_t first[EDIT_BINS] = {}, retry[EDIT_BINS] = {}, trace[EDIT_BINS] = {};
    for (size_t s = 0; s < b->slot_pair.size(); ++s) {
        const int n = b->rows[s], m = b->cols[s];
        const int start = b->start_bin[edit_length_class(std::max(n, m))];
        const int widest = std::max(start, edit_widest(n + m));
        for (int k = start; k <= widest; ++k) ++first[k];
        for (int k = start + 1; k <= widest; ++k) ++retry[k];
        for (int k = 0; k <= widest; ++k) ++trace[k];
    }
    for (int k = 0; k < EDIT_BINS; ++k) {
        b->first_count[k] = first[k];
        b->retry_reach[k] = retry[k];
        b->trace_reach[k] = trace[k];
    }
    for (int c = 0; c < EDIT_LENGTH_CLASSES; ++c) b->seeded_start[c] = b->start_bin[c];
    if (b->edit_graph) {
        (void)hipGraphExecDestroy(b->edit_graph);
        b->edit_graph = nullptr;
    }
}

// Learned seeds without leaving the device (unit-cost batches): features, the network's predictions and each
// pair's first band and queue, all on the batch's stream.
int64_t seed_unit_learned(dinara_batch *b, dinara_mlp *net, double margin, double slope) {
    const int64_t slots = (int64_t)b->slot_pair.size();
    if (slots == 0) return 0;
    DeviceContext *ctx = b->ctx;
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    (void)hipGetLastError();
    if (!b->features_d.reserve((size_t)slots * FEATURE_STRIDE * 4) || !b->predictions_d.reserve((size_t)slots * 4))
        return DINARA_OUT_OF_MEMORY;
    SweepArgs sa = sweep_args(b);
    launch_features(sa.tape, (int)slots, b->reversed ? 1 : 0, static_cast<float *>(b->features_d.ptr), ctx->stream);
    if (const int64_t code = mlp_predict_into(net, static_cast<const float *>(b->features_d.ptr), slots,
                                              static_cast<float *>(b->predictions_d.ptr)))
        return code;
    EditStart start{};
    for (int c = 0; c < EDIT_LENGTH_CLASSES; ++c) start.bin[c] = b->start_bin[c];
    start.bins = b->first_bins;
    launch_edit_seed(edit_args(b), static_cast<const float *>(b->predictions_d.ptr), margin, slope, start,
                     (int)slots, ctx->stream);
    seeded_shape(b);
    return hipPeekAtLastError() == hipSuccess ? 0 : DINARA_OUT_OF_MEMORY;
}

void drop_graph(dinara_batch *b) {
    if (b->edit_graph) {
        DeviceGuard guard(b->ctx);
        (void)hipGraphExecDestroy(b->edit_graph);
        b->edit_graph = nullptr;
    }
}

// Tunes the unit-cost sweep's launch shape on the batch itself: first the workgroups a compute unit, then each
// length class's least first bin (heaviest class first, widening while the first pass gets faster). Each
// candidate is timed as the faster of two first passes (no tracing).
int64_t autotune(dinara_batch *b, int64_t *chosen) {
    const int64_t slots = (int64_t)b->slot_pair.size();
    auto report = [&]() {
        if (!chosen) return;
        chosen[0] = b->grid_per_cu;
        for (int c = 0; c < EDIT_LENGTH_CLASSES; ++c) chosen[1 + c] = b->start_bin[c];
        chosen[1 + EDIT_LENGTH_CLASSES] = b->side_by_side_bins ? 1 : 0;
    };
    if (!b->unit || slots == 0) {
        report();
        return 0;
    }
    DeviceContext *ctx = b->ctx;
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    (void)hipGetLastError();
    int64_t failure = 0;
    auto measure = [&]() {
        double best = 1e300;
        for (int i = 0; i < 2; ++i) {
            if (const int64_t code = run_unit(b, false)) {
                failure = code;
                return 1e300;
            }
            best = std::min(best, b->run_ms);
        }
        return best;
    };
    double best = measure();
    int best_grid = b->grid_per_cu;
    for (int grid : {2, 4, 8, 16}) {
        if (grid == best_grid) continue;
        b->grid_per_cu = grid;
        drop_graph(b);
        const double t = measure();
        if (t < best) {
            best = t;
            best_grid = grid;
        }
    }
    b->grid_per_cu = best_grid;
    drop_graph(b);
    // The bins side by side or one after another.
    b->side_by_side_bins = !b->side_by_side_bins;
    drop_graph(b);
    if (const double t = measure(); t < best)
        best = t;
    else
        b->side_by_side_bins = !b->side_by_side_bins;
    drop_graph(b);
    // Queues the device filed from learned seeds keep their bands: the start bins stay.
    if (b->seeded_start[0] >= 0) {
        report();
        return failure;
    }
    // Length classes by weight (the sum of their pairs' squared longer sides), heaviest first.
    double weight[EDIT_LENGTH_CLASSES] = {};
    for (int64_t s = 0; s < slots; ++s) {
        const double longer = std::max(b->rows[s], b->cols[s]);
        weight[edit_length_class((int)longer)] += longer * longer;
    }
    int order[EDIT_LENGTH_CLASSES];
    std::iota(order, order + EDIT_LENGTH_CLASSES, 0);
    std::sort(order, order + EDIT_LENGTH_CLASSES, [&](int x, int y) { return weight[x] > weight[y]; });
    for (int c : order) {
        if (weight[c] == 0) continue;
        int best_start = b->start_bin[c];
        for (int start = best_start + 1; start < EDIT_BINS; ++start) {
            b->start_bin[c] = start;
            if (const int64_t code = unit_lists(b)) return code;
            const double t = measure();
            if (t >= best) break;
            best = t;
            best_start = start;
        }
        b->start_bin[c] = best_start;
        if (const int64_t code = unit_lists(b)) return code;
    }
    report();
    return failure;
}

}  // namespace

extern "C" {

int64_t dinara_batch_seed(dinara_batch *b, const int64_t *predicted) {
    if (!b) return DINARA_INVALID_MODE;
    return seed_slots(b, [&](int64_t s) { return predicted[b->slot_pair[s]]; });
}

int64_t dinara_batch_seed_learned(dinara_batch *b, dinara_mlp *net, double margin) {
    return dinara_batch_seed_learned_by_length(b, net, margin, 0.0);
}

int64_t dinara_batch_seed_learned_by_length(dinara_batch *b, dinara_mlp *net, double margin, double slope) {
    if (!b || !net) return DINARA_INVALID_MODE;
    if (b->unit) return seed_unit_learned(b, net, margin, slope);
    const int64_t slots = (int64_t)b->slot_pair.size();
    if (slots == 0) return 0;
    std::vector<float> predicted((size_t)slots);
    {
        DeviceContext *ctx = b->ctx;
        std::lock_guard<std::mutex> serial(ctx->lock);
        DeviceGuard guard(ctx);
        DeviceBuffer features;
        if (!features.reserve((size_t)slots * FEATURE_STRIDE * 4)) return DINARA_OUT_OF_MEMORY;
        SweepArgs a = sweep_args(b);
        launch_features(a.tape, (int)slots, b->reversed ? 1 : 0, static_cast<float *>(features.ptr), ctx->stream);
        if (hipPeekAtLastError() != hipSuccess) return DINARA_OUT_OF_MEMORY;
        if (const int64_t code = mlp_predict_device(net, static_cast<const float *>(features.ptr), slots,
                                                    predicted.data()))
            return code;
    }
    return seed_slots(b, [&](int64_t s) {
        const double longer = std::max(1000.0, (double)std::max(b->rows[s], b->cols[s]));
        const double guess = std::expm1((double)predicted[s] + margin + slope * std::log(longer / 1000.0));
        // Clamped before the cast: past 2^40 every band is the whole matrix anyway, and an infinite or huge
        // prediction must not reach a conversion it does not fit (NaN fails the test and gives 0).
        constexpr double most = 1099511627776.0;
        return guess > 0 ? (int64_t)(guess < most ? guess : most) : int64_t(0);
    });
}

int64_t dinara_batch_set_retry(dinara_batch *b, int64_t doubling) {
    if (!b) return DINARA_INVALID_MODE;
    const bool changed = b->doubling != (doubling != 0);
    b->doubling = doubling != 0;
    drop_graph(b);
    // The host-filed first queues follow the policy (doubling keeps to the powers of two); seeded ones are filed
    // again by the next seeding.
    if (!changed || !b->unit || b->slot_pair.empty()) return 0;
    std::lock_guard<std::mutex> serial(b->ctx->lock);
    DeviceGuard guard(b->ctx);
    return unit_lists(b);
}

int64_t dinara_batch_set_graph(dinara_batch *b, int64_t on) {
    if (!b) return DINARA_INVALID_MODE;
    b->use_graph = on != 0;
    return 0;
}

int64_t dinara_batch_set_keep_first(dinara_batch *b, int64_t on) {
    if (!b) return DINARA_INVALID_MODE;
    b->keep_first = on != 0;
    drop_graph(b);
    b->arena_bound = 0;  // the arena it asks for follows the setting: worked out again at the next run
    return 0;
}

int64_t dinara_batch_set_side_by_side(dinara_batch *b, int64_t on) {
    if (!b) return DINARA_INVALID_MODE;
    b->side_by_side_bins = on != 0;
    drop_graph(b);
    return 0;
}

int64_t dinara_batch_set_whole(dinara_batch *b, int64_t on) {
    if (!b || b->free_ends || b->user_band) return DINARA_INVALID_MODE;
    b->whole = on != 0;
    return 0;
}

int64_t dinara_batch_set_persistent(dinara_batch *b, int64_t on) {
    if (!b) return DINARA_INVALID_MODE;
    b->persistent = on != 0;
    drop_graph(b);
    return 0;
}

int64_t dinara_batch_set_tuning(dinara_batch *b, int64_t grid_per_cu, const int64_t *start_bins) {
    if (!b || grid_per_cu < 1 || grid_per_cu > 64) return DINARA_INVALID_MODE;
    if (start_bins)
        for (int c = 0; c < EDIT_LENGTH_CLASSES; ++c)
            if (start_bins[c] < 0 || start_bins[c] >= EDIT_BINS) return DINARA_INVALID_MODE;
    b->grid_per_cu = (int)grid_per_cu;
    if (start_bins)
        for (int c = 0; c < EDIT_LENGTH_CLASSES; ++c) b->start_bin[c] = (int)start_bins[c];
    drop_graph(b);
    if (!b->unit || b->slot_pair.empty()) return 0;
    std::lock_guard<std::mutex> serial(b->ctx->lock);
    DeviceGuard guard(b->ctx);
    return unit_lists(b);
}

int64_t dinara_batch_set_bins(dinara_batch *b, int64_t bins) {
    if (!b || bins <= 0 || bins > (int64_t)EDIT_ALL_BINS) return DINARA_INVALID_MODE;
    b->first_bins = (uint32_t)bins;
    drop_graph(b);
    // The host-filed first queues follow the set; seeded ones are filed again by the next seeding.
    if (!b->unit || b->slot_pair.empty()) return 0;
    std::lock_guard<std::mutex> serial(b->ctx->lock);
    DeviceGuard guard(b->ctx);
    return unit_lists(b);
}

int64_t dinara_batch_autotune(dinara_batch *b, int64_t *chosen) {
    if (!b) return DINARA_INVALID_MODE;
    return autotune(b, chosen);
}

void dinara_batch_free(dinara_batch *batch) {
    if (!batch) return;
    {
        DeviceGuard guard(batch->ctx);
        delete batch;
    }
}

double dinara_batch_stat(dinara_batch *b, int64_t what) {
    if (!b) return 0;
    const bool counted = what == 4 || what == 9 ||
                         (what >= 700 && what < 1200 && what / 100 != 8 && what % 100 < EDIT_BINS);
    if (counted && b->stats_pending) {  // the unit path's counters of the last run
        DeviceContext *ctx = b->ctx;
        std::lock_guard<std::mutex> serial(ctx->lock);
        DeviceGuard guard(ctx);
        uint32_t stats[2 * EDIT_BINS + 2] = {};
        unsigned long long work[2 * EDIT_BINS] = {};
        if (b->edit_stats.read(ctx, stats, sizeof(stats)) && b->edit_work.read(ctx, work, sizeof(work))) {
            for (int bin = 0; bin < EDIT_BINS; ++bin) {
                b->edit_sweeps[bin] = stats[bin];
                b->trace_sweeps[bin] = stats[EDIT_BINS + bin];
                b->sweep_work[bin] = (double)work[bin];
                b->trace_work[bin] = (double)work[EDIT_BINS + bin];
            }
            b->first_proven = (double)(b->stats_slots - stats[2 * EDIT_BINS]);
            b->walked_first = stats[2 * EDIT_BINS + 1];
        }
        b->stats_pending = false;
    }
    switch (what) {
        case 0: return b->run_ms;
        case 1: return b->sweep_ms;
        case 2: return b->launches;
        case 4: return b->first_proven;
        case 5: return b->walk_ms;
        case 6: return b->unit ? 1 : 0;
        case 7: return b->graph_used;
        case 8: return b->trace_passes;
        case 9: return b->walked_first;
        case 10: return b->full_pairs;
        case 11: return b->full_ms;
        case 12: return EDIT_BINS;
        case 13: return b->first_bins;
        case 14: return b->group16_top;
        default: break;
    }
    if (what >= 600 && what < 1300 && what % 100 < EDIT_BINS) {
        const int bin = (int)(what % 100);
        switch (what / 100) {
            case 12: return edit_width(bin);
            case 10: return b->sweep_work[bin];
            case 11: return b->trace_work[bin];
            case 6: return b->edit_ms[bin];
            case 7: return b->edit_sweeps[bin];
            case 8: return b->trace_ms[bin];
            case 9: return b->trace_sweeps[bin];
        }
    }
    if (what >= 100 && what < 500 && what % 100 < CLASSES) {
        const int c = (int)(what % 100);
        switch (what / 100) {
            case 1: return b->class_ms[c];
            case 2: return b->class_launches[c];
            case 4: return b->class_pairs[c];
        }
    }
    switch (what) {
        default: return 0;
    }
}

// A batch run once (the drop-in calls): the unit path's launches go one by one without timing events, since a
// captured graph would be instantiated for a single replay.
void one_shot(dinara_batch *b) {
    if (!b->unit) return;
    b->use_graph = false;
    b->timed = false;
}

int64_t dinara_gpu_distances(int64_t gpu, int64_t pairs, const char *const *references,
                             const int64_t *reference_lengths, const char *const *queries,
                             const int64_t *query_lengths, const dinara_costs *costs, const dinara_mode *mode,
                             const dinara_options *options, int64_t threads, int64_t *results) {
    ParsedCosts parsed = parse_costs(costs);
    if (parsed.code) return parsed.code;
    if (const int64_t code = check_mode(mode)) return code;
    if (pairs <= 0) return 0;
    int64_t status = 0;
    dinara_batch *b = batch_new(gpu, DINARA_BATCH_DISTANCES, pairs, references, reference_lengths, queries,
                                query_lengths, costs, mode, options, threads, &status);
    if (!b) return status;
    one_shot(b);
    int64_t code = run(b);
    if (code == 0) code = dinara_batch_distances(b, results);
    dinara_batch_free(b);
    return code;
}

int64_t dinara_gpu_alignments(int64_t gpu, int64_t pairs, const char *const *references,
                              const int64_t *reference_lengths, const char *const *queries,
                              const int64_t *query_lengths, const dinara_costs *costs, const dinara_mode *mode,
                              const dinara_options *options, int64_t threads, dinara_alignment *alignments,
                              int64_t *statuses) {
    ParsedCosts parsed = parse_costs(costs);
    if (parsed.code) return parsed.code;
    if (const int64_t code = check_mode(mode)) return code;
    if (pairs <= 0) return 0;
    int64_t status = 0;
    dinara_batch *b = batch_new(gpu, DINARA_BATCH_ALIGNMENTS, pairs, references, reference_lengths, queries,
                                query_lengths, costs, mode, options, threads, &status);
    if (!b) return status;
    one_shot(b);
    int64_t code = run(b);
    if (code == 0) code = dinara_batch_alignments(b, alignments, statuses);
    dinara_batch_free(b);
    return code;
}

int64_t dinara_distances(int64_t pairs, const char *const *references, const int64_t *reference_lengths,
                         const char *const *queries, const int64_t *query_lengths, const dinara_costs *costs,
                         const dinara_mode *mode, const dinara_options *options, int64_t threads, int64_t *results) {
    return dinara_gpu_distances(0, pairs, references, reference_lengths, queries, query_lengths, costs, mode, options,
                                threads, results);
}

int64_t dinara_alignments(int64_t pairs, const char *const *references, const int64_t *reference_lengths,
                          const char *const *queries, const int64_t *query_lengths, const dinara_costs *costs,
                          const dinara_mode *mode, const dinara_options *options, int64_t threads,
                          dinara_alignment *alignments, int64_t *statuses) {
    return dinara_gpu_alignments(0, pairs, references, reference_lengths, queries, query_lengths, costs, mode,
                                 options, threads, alignments, statuses);
}

}  // extern "C"

namespace dinara {

// dinara_gpu_distances under unit costs with every device buffer taken from `carve` (see carved.h).
int64_t carved_unit_distances(Carve *carve, int64_t gpu, int64_t pairs, const char *const *references,
                              const int64_t *reference_lengths, const char *const *queries,
                              const int64_t *query_lengths, const dinara_costs *costs, const dinara_mode *mode,
                              const dinara_options *options, int64_t threads, int64_t *results) {
    ParsedCosts parsed = parse_costs(costs);
    if (parsed.code) return parsed.code;
    if (const int64_t code = check_mode(mode)) return code;
    if (parsed.two_piece || free_mode(mode)) return DINARA_INVALID_MODE;
    const Options o = parse_options(options);
    const bool unit = parsed.opening == 0 && parsed.del_opening == 0 && parsed.extension == parsed.mismatch &&
                      parsed.del_extension == parsed.mismatch && o.band_low <= -UNBOUNDED && o.band_high >= UNBOUNDED;
    if (!unit) return DINARA_INVALID_MODE;
    if (pairs <= 0) return 0;
    CarveScope scope(carve);
    int64_t status = 0;
    dinara_batch *b = batch_new(gpu, DINARA_BATCH_DISTANCES, pairs, references, reference_lengths, queries,
                                query_lengths, costs, mode, options, threads, &status);
    if (!b) return carve->exhausted ? DINARA_SCRATCH_FULL : status;
    int64_t code = 0;
    if (!b->unit) {
        code = DINARA_INVALID_MODE;  // the bit-parallel path switched off
    } else {
        // One stream, launches one by one: no graph to instantiate, no side streams or timing events to make.
        b->use_graph = false;
        b->one_stream = true;
        b->timed = false;
        code = run(b);
        if (code == 0) code = dinara_batch_distances(b, results);
        if (code != 0 && carve->exhausted) code = DINARA_SCRATCH_FULL;
    }
    dinara_batch_free(b);
    return code;
}

}  // namespace dinara
