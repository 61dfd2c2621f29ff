// The C ABI's substitution-table calls: scores and alignments under a `dinara_scoring`, global or local, on the
// device. Reference behaviour followed: scoring.mojo:126-238 (the table, gaps and 32-bit reach), common.mojo:267-289
// (letters to codes), api.mojo:843-1001 (the batch calls and their modes), scoring.mojo:544-560 (a local
// alignment: its end, its start, the letters between aligned globally) and :724-745 (spans by rfind).
//
// A batch is validated and packed once, then its passes run on the device: scores take one sweep; a global
// alignment a sweep that keeps every decision and a walk back; a local alignment the best end, the reach back to
// its start, and the span's global alignment with its walk.

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "../../include/dinara.h"
#include "device.h"
#include "host.h"
#include "score.h"

using namespace dinara;

namespace {

constexpr uint8_t UNKNOWN_LETTER = 0xFF;

// A device step that failed: DINARA_OUT_OF_MEMORY, and with DINARA_DEBUG set in the environment a line on stderr
// naming the step and the runtime's last error.
int64_t failed(const char *step) {
    if (std::getenv("DINARA_DEBUG")) {
        const hipError_t e = hipGetLastError();
        std::fprintf(stderr, "dinara: %s failed (%s)\n", step, hipGetErrorString(e));
    }
    return DINARA_OUT_OF_MEMORY;
}
constexpr int64_t INT32_TOP = 0x7fffffff;

// A Scoring checked as the reference checks one (scoring.mojo:200-214, gotoh.mojo:47-54): 1 to 32 letters, no
// '-', a table, a gap's parts zero or less and within 32 bits. `code` is nonzero when the batch fails whole.
struct ParsedScoring {
    int64_t code = 0;
    int letters = 0;
    uint8_t codes[256];
    int8_t table[32 * 32];
    int open = 0, extend = 0;  // a gap's first letter (opening + extension), each later one
    int64_t reach_opening = 0, reach_step = 0;
};

ParsedScoring parse_scoring(const dinara_scoring *s) {
    ParsedScoring p;
    std::memset(p.codes, UNKNOWN_LETTER, sizeof p.codes);
    std::memset(p.table, 0, sizeof p.table);
    if (!s || !s->alphabet || !s->table || s->letters < 1 || s->letters > 32) {
        p.code = DINARA_INVALID_COSTS;
        return p;
    }
    p.letters = (int)s->letters;
    for (int i = 0; i < p.letters; ++i) {
        const uint8_t byte = (uint8_t)s->alphabet[i];
        if (byte == '-') {
            p.code = DINARA_INVALID_COSTS;
            return p;
        }
        p.codes[byte] = (uint8_t)i;  // a repeated letter takes its last place
    }
    if (s->opening > 0 || s->extension > 0 || std::min(s->opening, s->extension) < -INT32_TOP ||
        s->opening + s->extension < -INT32_TOP) {
        p.code = DINARA_INVALID_COSTS;
        return p;
    }
    int best = -128, least = 127;
    for (int a = 0; a < p.letters; ++a)
        for (int b = 0; b < p.letters; ++b) {
            const int8_t v = s->table[a * p.letters + b];
            p.table[a * 32 + b] = v;
            best = std::max<int>(best, v);
            least = std::min<int>(least, v);
        }
    p.open = (int)(s->opening + s->extension);
    p.extend = (int)s->extension;
    p.reach_opening = 2 * -(int64_t)p.open;
    p.reach_step = std::max<int64_t>(std::max<int64_t>(best, -least), -(int64_t)p.extend);
    return p;
}

// Whether a pair's scores stay well inside 32 bits (reference scoring.mojo:216-238, ScoreReach.check).
bool within_reach(const ParsedScoring &p, int64_t rows, int64_t cols, bool floored) {
    const int64_t letters = floored ? std::min(rows, cols) : rows + cols;
    return p.reach_opening + 2 * (letters + 2) * p.reach_step < (int64_t(1) << 28);
}

// Global or local (reference api.mojo:853-866): a mode's own match score must be zero; other modes have no device
// path here.
int64_t check_scoring_mode(const dinara_mode *m, bool *local) {
    *local = false;
    if (!m) return 0;
    if (m->match_score != 0) return DINARA_INVALID_MODE;
    if (m->kind == DINARA_LOCAL) {
        *local = true;
        return 0;
    }
    if (m->kind != DINARA_ENDS_FREE) return DINARA_INVALID_MODE;
    if ((m->reference_start | m->reference_end | m->query_start | m->query_end) != 0) return DINARA_INVALID_MODE;
    return 0;
}

int64_t gap_run(const ParsedScoring &p, int64_t letters) {
    return letters == 0 ? 0 : p.open + (letters - 1) * (int64_t)p.extend;
}

// Whether a pair of a pass of `pairs` takes a quarter wave: it holds the pair and its staged reference, and the pass is
// large enough that sharing a wave pays. Whole waves' chains are shorter (148 columns: 3 a lane rather than 10) but
// there are four times as many. Scores of a pass, quarters against wholes: 256 pairs of 60 letters 14 to 16 us; of 148
// letters 34 to 31 at 1,000 pairs, 37 to 44 at 1,500; of 240 residues 89 to 71 at 2,000, 89 to 93 at 3,000.
bool takes_quarter(int64_t pairs, int64_t rows, int64_t cols) {
    return cols <= SCORE_NARROW_COLS && rows + 4 <= SCORE_RING && cols * cols <= 16 * pairs;
}

// The last place `needle` occurs in `hay` (reference scoring.mojo:734-735, String.rfind over bytes).
// Eight bytes are compared before the call that compares them all.
int64_t rfind(const char *hay, int64_t n, const char *needle, int64_t k) {
    if (k == 0) return 0;
    uint64_t head = 0, there = 0;
    if (k >= 8) std::memcpy(&head, needle, 8);
    for (int64_t at = n - k; at >= 0; --at) {
        if (k >= 8) std::memcpy(&there, hay + at, 8);
        if (there == head && std::memcmp(hay + at, needle, (size_t)k) == 0) return at;
    }
    return -1;
}

}  // namespace

// ------------------------------------------------------------------ the batch

struct ScoreLaunch {
    ScoreArgs args;
    size_t lds;
};

struct dinara_scoring_batch {
    int gpu = 0;
    int64_t kind = DINARA_BATCH_DISTANCES;  // DISTANCES: scores; ALIGNMENTS: alignments
    bool local = false;
    int eqx = 1;
    int64_t pairs = 0;
    int64_t threads = 0;
    ParsedScoring scoring;
    DeviceContext *ctx = nullptr;
    const char *const *refs = nullptr;  // the caller's letters, for spans (valid during the call that made it)
    const char *const *qrys = nullptr;
    std::vector<int64_t> code;          // per pair: 0 on the device, else its own result code or a settled host value
    std::vector<int64_t> rows, cols;
    std::vector<int32_t> slot_pair;     // slot -> pair, the pairs the device takes, longest first
    std::vector<int64_t> host_score;    // per pair: a score settled without the device (an empty side)
    std::vector<int32_t> view_h;        // per slot: reference begin, letters, query begin, letters
    std::vector<int32_t> score_h, end_row_h, end_col_h, reach_row_h, reach_col_h, cigar_length_h;
    std::vector<int64_t> cigar_offset_h;
    std::vector<char> cigars_h;
    // device memory
    DeviceBuffer codes, ref_at, qry_at, view, list, table, score, end_row, end_col, target, walk_base, walk_columns, arena,
        arena_at, carry, carry_at, op_scratch, op_base, cigars, cigar_used, cigar_offset, cigar_length;
    // timing of the last run
    double run_ms = 0, pass_ms[4] = {0, 0, 0, 0};
    int launches = 0;
    bool ran = false;
    // A global batch's one pass, laid out by its first run: its views are its whole pairs, at every run the same.
    bool planned = false;
    std::vector<ScoreLaunch> plan;
    Region region;  // what most of the buffers lie in
    ~dinara_scoring_batch() {
        if (region.base) give_back(ctx, region);
    }
};

namespace {

using Batch = dinara_scoring_batch;

ScoreArgs score_args(Batch *b, int mode, int reversed) {
    ScoreArgs a{};
    a.codes = static_cast<const uint8_t *>(b->codes.ptr);
    a.ref_at = static_cast<const int64_t *>(b->ref_at.ptr);
    a.qry_at = static_cast<const int64_t *>(b->qry_at.ptr);
    a.view = static_cast<const int32_t *>(b->view.ptr);
    a.reversed = reversed;
    a.table = static_cast<const int8_t *>(b->table.ptr);
    a.letters = b->scoring.letters;
    a.open = b->scoring.open;
    a.extend = b->scoring.extend;
    a.mode = mode;
    a.score = static_cast<int32_t *>(b->score.ptr);
    a.end_row = static_cast<int32_t *>(b->end_row.ptr);
    a.end_col = static_cast<int32_t *>(b->end_col.ptr);
    a.target = static_cast<const int32_t *>(b->target.ptr);
    a.walk_base = static_cast<uint64_t *>(b->walk_base.ptr);
    a.walk_columns = static_cast<int32_t *>(b->walk_columns.ptr);
    a.eqx = b->eqx;
    a.op_scratch = static_cast<char *>(b->op_scratch.ptr);
    a.op_base = static_cast<const int64_t *>(b->op_base.ptr);
    a.cigars = static_cast<char *>(b->cigars.ptr);
    a.cigar_used = static_cast<unsigned long long *>(b->cigar_used.ptr);
    a.cigar_offset = static_cast<int64_t *>(b->cigar_offset.ptr);
    a.cigar_length = static_cast<int32_t *>(b->cigar_length.ptr);
    a.slots = (int)b->slot_pair.size();
    return a;
}

// The table's best score (at least 0).
int top_score(const Batch *b) {
    int top = 0;
    for (int x = 0; x < b->scoring.letters; ++x)
        for (int y = 0; y < b->scoring.letters; ++y) top = std::max<int>(top, b->scoring.table[x * 32 + y]);
    return top;
}

// Whether scores may be held less `extend` a row and a column: the raised letters' scores still fit their bytes.
bool extensions_free(const Batch *b) {
    int top = -128;
    for (int x = 0; x < b->scoring.letters; ++x)
        for (int y = 0; y < b->scoring.letters; ++y) top = std::max<int>(top, b->scoring.table[x * 32 + y]);
    return top - 2 * (int64_t)b->scoring.extend <= 127;
}

// Lays one pass out over the slots whose views are not empty: the pairs that take a whole wave in one launch, those that
// take a quarter in another (or more, when a trace's decisions pass the budget).
int64_t plan_pass(Batch *b, int mode, int reversed, const std::vector<int32_t> &slots, std::vector<ScoreLaunch> &out) {
    DeviceContext *ctx = b->ctx;
    const int32_t *view = b->view_h.data();
    const bool shifted = mode != SCORE_LOCAL && extensions_free(b);
    auto rows_of = [&](int32_t s) { return (int64_t)view[4 * s + 1]; };
    auto cols_of = [&](int32_t s) { return (int64_t)view[4 * s + 3]; };
    out.clear();
    const bool quarters = shifted && (mode == SCORE_GLOBAL || mode == SCORE_TRACE);
    std::vector<int32_t> all, narrow;  // the whole-wave pairs, then the quarter-wave pairs
    all.reserve(slots.size());
    for (int32_t s : slots) {
        if (rows_of(s) <= 0 || cols_of(s) <= 0) continue;
        if (quarters && takes_quarter((int64_t)slots.size(), rows_of(s), cols_of(s))) narrow.push_back(s);
        else all.push_back(s);
    }
    const int64_t wide = (int64_t)all.size();
    // Pairs that share a wave are of a size; whole views come sorted.
    if (b->local)
        std::stable_sort(narrow.begin(), narrow.end(),
                         [&](int32_t x, int32_t y) { return rows_of(x) * cols_of(x) > rows_of(y) * cols_of(y); });
    all.insert(all.end(), narrow.begin(), narrow.end());
    if (all.empty()) return 0;
    // Each wave's place among the kept columns and its launch's decisions, by its largest pair.
    std::vector<int64_t> carry_at, arena_at;
    std::vector<size_t> first_wave;  // of each launch
    std::vector<int64_t> first_pair;
    int64_t carry = 0, most_carry = 0, decisions = 0, most_decisions = 0;  // of a launch, and the most of one
    for (int kind = 0; kind < 2; ++kind) {
        const int64_t begin = kind == 0 ? 0 : wide, end = kind == 0 ? wide : (int64_t)all.size();
        if (begin == end) continue;
        ScoreArgs a = score_args(b, mode, reversed);
        a.shifted = shifted;
        a.lanes = kind == 0 ? 64 : SCORE_NARROW;
        const int64_t pairs = 64 / a.lanes;
        int64_t rows_max = 0, shorter = 0;
        for (int64_t i = begin; i < end; ++i) {
            rows_max = std::max(rows_max, rows_of(all[i]));
            shorter = std::max(shorter, std::min(rows_of(all[i]), cols_of(all[i])));
        }
        a.ref_room = (int)std::min<int64_t>(SCORE_RING, (rows_max + 4 + 3) & ~int64_t(3));
        // A local end's key: the rows' bits below a score no greater than the table's best times the shorter side.
        if (mode == SCORE_LOCAL) {
            int bits = 1;
            while (bits < 31 && (int64_t(1) << bits) <= rows_max) ++bits;
            if ((int64_t)top_score(b) * shorter < (int64_t(1) << (32 - bits))) a.end_bits = bits;
        }
        const size_t launches = out.size();
        size_t lds = 0;
        for (int64_t at = begin; at < end; at += pairs) {
            int64_t rows = 0, cols = 0;
            for (int64_t i = at; i < std::min(end, at + pairs); ++i) {
                rows = std::max(rows, rows_of(all[i]));
                cols = std::max(cols, cols_of(all[i]));
            }
            lds = std::max(lds, score_lds(b->scoring.letters, a.lanes, (int)cols, a.ref_room));
            const int64_t words = mode == SCORE_TRACE ? score_decisions(a.lanes, rows, cols) : 0;
            if (at == begin || (decisions > 0 && (decisions + words) * 4 > (int64_t)ARENA_BUDGET)) {
                carry = decisions = 0;
                out.push_back({a, 0});
                first_wave.push_back(carry_at.size());
                first_pair.push_back(at);
            }
            out.back().args.count += (int)(std::min(end, at + pairs) - at);
            carry_at.push_back(carry);
            carry += score_carry(a.lanes, rows, cols);
            most_carry = std::max(most_carry, carry);
            arena_at.push_back(decisions);
            decisions += words;
            most_decisions = std::max(most_decisions, decisions);
        }
        for (size_t l = launches; l < out.size(); ++l) out[l].lds = lds;
    }
    if (!b->list.upload(ctx, all.data(), all.size() * 4)) return failed("list upload");
    if (most_carry > 0 && (!b->carry.reserve((size_t)most_carry * 4) ||
                           !b->carry_at.upload(ctx, carry_at.data(), carry_at.size() * 8)))
        return failed("carry");
    if (mode == SCORE_TRACE && (!b->arena.reserve((size_t)most_decisions * 4) ||
                                !b->arena_at.upload(ctx, arena_at.data(), arena_at.size() * 8)))
        return failed("arena");
    for (size_t l = 0; l < out.size(); ++l) {
        ScoreArgs &a = out[l].args;
        a.list = static_cast<const int32_t *>(b->list.ptr) + first_pair[l];
        if (most_carry > 0) {
            a.carry = static_cast<int32_t *>(b->carry.ptr);
            a.carry_at = static_cast<const int64_t *>(b->carry_at.ptr) + first_wave[l];
        }
        if (mode == SCORE_TRACE) {
            a.arena = static_cast<uint32_t *>(b->arena.ptr);
            a.arena_at = static_cast<const int64_t *>(b->arena_at.ptr) + first_wave[l];
        }
    }
    return 0;
}

// One pass as planned, each trace launch followed by its walk.
int64_t run_pass(Batch *b, const std::vector<ScoreLaunch> &plan, hipEvent_t start, hipEvent_t stop, double *pass_ms) {
    DeviceContext *ctx = b->ctx;
    if (plan.empty()) return 0;
    hipEventRecord(start, ctx->stream);
    for (const ScoreLaunch &launch : plan) {
        launch_score(launch.args, launch.lds, ctx->stream);
        if (hipPeekAtLastError() != hipSuccess) return failed("score launch");
        b->launches += 1;
        if (launch.args.mode == SCORE_TRACE) {
            launch_score_walk(launch.args, ctx->stream);
            if (hipPeekAtLastError() != hipSuccess) return failed("walk launch");
        }
    }
    hipEventRecord(stop, ctx->stream);
    if (hipEventSynchronize(stop) != hipSuccess) return failed("pass");
    float ms = 0;
    hipEventElapsedTime(&ms, start, stop);
    *pass_ms += ms;
    return 0;
}

int64_t prepare(Batch *b, const char *const *refs, const int64_t *ref_lens, const char *const *qrys,
                const int64_t *qry_lens) {
    DeviceContext *ctx = b->ctx;
    const int64_t pairs = b->pairs;
    b->code.assign(pairs, 0);
    b->rows.assign(pairs, 0);
    b->cols.assign(pairs, 0);
    b->host_score.assign(pairs, 0);
    parallel_for(pairs, b->threads, [&](int64_t lo, int64_t hi) {
        for (int64_t i = lo; i < hi; ++i) {
            const int64_t n = ref_lens[i], m = qry_lens[i];
            if (n < 0 || m < 0) {
                b->code[i] = DINARA_INVALID_LENGTH;
                continue;
            }
            b->rows[i] = n;
            b->cols[i] = m;
            bool known = true;
            for (int64_t k = 0; k < n && known; ++k) known = b->scoring.codes[(uint8_t)refs[i][k]] != UNKNOWN_LETTER;
            for (int64_t k = 0; k < m && known; ++k) known = b->scoring.codes[(uint8_t)qrys[i][k]] != UNKNOWN_LETTER;
            if (!known) {
                b->code[i] = DINARA_UNSUPPORTED_SYMBOLS;
                continue;
            }
            if (!within_reach(b->scoring, n, m, b->local) || n >= (int64_t(1) << 20) || m >= (int64_t(1) << 20)) {
                b->code[i] = DINARA_INVALID_COSTS;
                continue;
            }
            // Against an empty side: one gap of every letter, or no local alignment (reference
            // scoring.mojo:384-396).
            if (n == 0 || m == 0) b->code[i] = 1, b->host_score[i] = b->local ? 0 : gap_run(b->scoring, n + m);
        }
    });
    b->slot_pair.clear();
    for (int64_t i = 0; i < pairs; ++i)
        if (b->code[i] == 0) b->slot_pair.push_back((int32_t)i);
    std::stable_sort(b->slot_pair.begin(), b->slot_pair.end(), [&](int32_t x, int32_t y) {
        return b->rows[x] * b->cols[x] > b->rows[y] * b->cols[y];
    });
    const int64_t slots = (int64_t)b->slot_pair.size();
    std::vector<int64_t> ref_at(std::max<int64_t>(slots, 1)), qry_at(std::max<int64_t>(slots, 1)), op_base(slots + 1);
    int64_t total = 0, ops = 0, text = 0;
    for (int64_t s = 0; s < slots; ++s) {
        const int32_t p = b->slot_pair[s];
        ref_at[s] = total;
        total += b->rows[p];
        qry_at[s] = total;
        total += b->cols[p];
        op_base[s] = ops;
        ops += 8 * ((b->rows[p] + b->cols[p]) / 32 + 1);
        text += 2 * (b->rows[p] + b->cols[p]) + 2;
    }
    op_base[slots] = ops;
    std::vector<uint8_t> codes((size_t)std::max<int64_t>(total, 1));
    parallel_for(slots, b->threads, [&](int64_t lo, int64_t hi) {
        for (int64_t s = lo; s < hi; ++s) {
            const int32_t p = b->slot_pair[s];
            for (int64_t k = 0; k < b->rows[p]; ++k) codes[ref_at[s] + k] = b->scoring.codes[(uint8_t)refs[p][k]];
            for (int64_t k = 0; k < b->cols[p]; ++k) codes[qry_at[s] + k] = b->scoring.codes[(uint8_t)qrys[p][k]];
        }
    });
    b->view_h.assign(4 * std::max<int64_t>(slots, 1), 0);
    const size_t n4 = (size_t)std::max<int64_t>(slots, 1) * 4;
    // The batch's buffers in one block, as far as it goes; what a run needs besides is allocated apart.
    Carve carve;
    b->region = ctx->take_region(codes.size() + 24 * n4 + ops + text + (64 << 10));
    std::optional<CarveScope> scope;
    if (b->region.base) {
        carve.base = b->region.base;
        carve.size = b->region.size;
        carve.image = b->region.image;
        carve.strict = false;
        scope.emplace(&carve);
    }
    if (!b->codes.upload(ctx, codes.data(), codes.size()) ||
        !b->ref_at.upload(ctx, ref_at.data(), ref_at.size() * 8) ||
        !b->qry_at.upload(ctx, qry_at.data(), qry_at.size() * 8) ||
        !b->table.upload(ctx, b->scoring.table, sizeof b->scoring.table) || !b->view.reserve(4 * n4) ||
        !b->score.reserve(n4) || !b->end_row.reserve(n4) || !b->end_col.reserve(n4) || !b->target.reserve(n4))
        return DINARA_OUT_OF_MEMORY;
    if (b->kind == DINARA_BATCH_ALIGNMENTS) {
        if (!b->walk_base.reserve(n4 * 2) || !b->walk_columns.reserve(n4) ||
            !b->op_base.upload(ctx, op_base.data(), op_base.size() * 8) ||
            !b->op_scratch.reserve(std::max<int64_t>(ops, 8)) || !b->cigars.reserve(std::max<int64_t>(text, 1)) ||
            !b->cigar_used.reserve(8) || !b->cigar_offset.reserve(n4 * 2) || !b->cigar_length.reserve(n4))
            return DINARA_OUT_OF_MEMORY;
    }
    return carve.flush(ctx) ? 0 : DINARA_OUT_OF_MEMORY;
}

// Sets every slot's view: both sequences whole, forward.
void whole_views(Batch *b) {
    for (size_t s = 0; s < b->slot_pair.size(); ++s) {
        const int32_t p = b->slot_pair[s];
        int32_t *v = &b->view_h[4 * s];
        v[0] = 0;
        v[1] = (int32_t)b->rows[p];
        v[2] = 0;
        v[3] = (int32_t)b->cols[p];
    }
}

bool read_slots(Batch *b, DeviceBuffer &buffer, std::vector<int32_t> &out) {
    out.resize(std::max<size_t>(b->slot_pair.size(), 1));
    return buffer.read(b->ctx, out.data(), out.size() * 4);
}

int64_t run(Batch *b) {
    DeviceContext *ctx = b->ctx;
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    b->launches = 0;
    b->run_ms = 0;
    for (double &ms : b->pass_ms) ms = 0;
    const size_t slots = b->slot_pair.size();
    b->ran = true;
    if (slots == 0) return 0;
    (void)hipGetLastError();  // an earlier, unrelated call's error is not this run's
    hipEvent_t start = ctx->event(0), stop = ctx->event(1), begin = ctx->event(2), end = ctx->event(3);
    hipEventRecord(begin, ctx->stream);
    std::vector<int32_t> all;
    if (!b->planned) {
        all.resize(slots);
        for (size_t s = 0; s < slots; ++s) all[s] = (int32_t)s;
        whole_views(b);
        if (!b->view.write(ctx, b->view_h.data(), b->view_h.size() * 4)) return failed("views");
    }
    const bool align = b->kind == DINARA_BATCH_ALIGNMENTS;
    if (align) hipMemsetAsync(b->cigar_used.ptr, 0, 8, ctx->stream);
    int64_t code = 0;
    if (!b->local) {
        if (!b->planned) code = plan_pass(b, align ? SCORE_TRACE : SCORE_GLOBAL, 0, all, b->plan);
        b->planned = code == 0;
        if (code == 0) code = run_pass(b, b->plan, start, stop, &b->pass_ms[align ? 3 : 0]);
    } else {
        std::vector<ScoreLaunch> plan;
        code = plan_pass(b, SCORE_LOCAL, 0, all, plan);
        if (code == 0) code = run_pass(b, plan, start, stop, &b->pass_ms[1]);
        if (code == 0 && align) {
            // The reach back from every local end above zero, over both prefixes reversed (reference
            // vector_score.mojo:37-162), then the span between start and end aligned globally.
            if (!read_slots(b, b->score, b->score_h) || !read_slots(b, b->end_row, b->end_row_h) ||
                !read_slots(b, b->end_col, b->end_col_h))
                return failed("local ends");
            std::vector<int32_t> reaching;
            for (size_t s = 0; s < slots; ++s) {
                int32_t *v = &b->view_h[4 * s];
                if (b->score_h[s] > 0) {
                    v[0] = 0;
                    v[1] = b->end_row_h[s];
                    v[2] = 0;
                    v[3] = b->end_col_h[s];
                    reaching.push_back((int32_t)s);
                } else {
                    v[1] = v[3] = 0;
                }
            }
            if (!b->view.write(ctx, b->view_h.data(), b->view_h.size() * 4) ||
                !b->target.write(ctx, b->score_h.data(), slots * 4))
                return failed("reach views");
            code = plan_pass(b, SCORE_REACH, 1, reaching, plan);
            if (code == 0) code = run_pass(b, plan, start, stop, &b->pass_ms[2]);
            if (code == 0) {
                if (!read_slots(b, b->end_row, b->reach_row_h) || !read_slots(b, b->end_col, b->reach_col_h))
                    return failed("reach starts");
                for (int32_t s : reaching) {
                    int32_t *v = &b->view_h[4 * s];
                    const int32_t er = b->end_row_h[s], ec = b->end_col_h[s];
                    const int32_t sr = b->reach_row_h[s] ? er - b->reach_row_h[s] : 0;
                    const int32_t sc = b->reach_row_h[s] ? ec - b->reach_col_h[s] : 0;
                    v[0] = sr;
                    v[1] = er - sr;
                    v[2] = sc;
                    v[3] = ec - sc;
                }
                if (!b->view.write(ctx, b->view_h.data(), b->view_h.size() * 4)) return failed("trace views");
                code = plan_pass(b, SCORE_TRACE, 0, reaching, plan);
                if (code == 0) code = run_pass(b, plan, start, stop, &b->pass_ms[3]);
            }
        }
    }
    hipEventRecord(end, ctx->stream);
    if (hipEventSynchronize(end) != hipSuccess) return failed("run");
    float ms = 0;
    hipEventElapsedTime(&ms, begin, end);
    b->run_ms = ms;
    return code;
}

int64_t fetch(Batch *b) {
    const size_t slots = b->slot_pair.size();
    if (slots == 0) return 0;
    if (!read_slots(b, b->score, b->score_h)) return failed("scores");
    if (b->kind == DINARA_BATCH_ALIGNMENTS) {
        uint64_t used = 0;
        b->cigar_offset_h.resize(slots);
        b->cigar_length_h.resize(slots);
        if (!b->cigar_used.read(b->ctx, &used, 8) ||
            !b->cigar_offset.read(b->ctx, b->cigar_offset_h.data(), slots * 8) ||
            !b->cigar_length.read(b->ctx, b->cigar_length_h.data(), slots * 4))
            return failed("cigar offsets");
        b->cigars_h.resize(std::max<uint64_t>(used, 1));
        if (used > b->cigars.size) {
            if (std::getenv("DINARA_DEBUG"))
                std::fprintf(stderr, "dinara: CIGARs claim %llu bytes of %zu\n", (unsigned long long)used, b->cigars.size);
            return DINARA_OUT_OF_MEMORY;
        }
        if (used > 0 && !b->cigars.read(b->ctx, b->cigars_h.data(), used)) return failed("cigars");
    }
    return 0;
}

Batch *batch_new(int64_t gpu, int64_t kind, int64_t pairs, const char *const *refs, const int64_t *ref_lens,
                 const char *const *qrys, const int64_t *qry_lens, const dinara_scoring *scoring,
                 const dinara_mode *mode, int64_t eqx, int64_t threads, int64_t *status) {
    auto fail = [&](int64_t code) -> Batch * {
        if (status) *status = code;
        return nullptr;
    };
    ParsedScoring parsed = parse_scoring(scoring);
    if (parsed.code) return fail(parsed.code);
    bool local = false;
    if (const int64_t code = check_scoring_mode(mode, &local)) return fail(code);
    if (kind != DINARA_BATCH_DISTANCES && kind != DINARA_BATCH_ALIGNMENTS) return fail(DINARA_INVALID_MODE);
    DeviceContext *ctx = device_context(gpu);
    if (!ctx) return fail(DINARA_NO_DEVICE);
    auto *b = new Batch();
    b->gpu = (int)gpu;
    b->ctx = ctx;
    b->kind = kind;
    b->local = local;
    b->eqx = eqx != 0;
    b->pairs = std::max<int64_t>(pairs, 0);
    b->threads = threads;
    b->scoring = parsed;
    b->refs = refs;
    b->qrys = qrys;
    int64_t code;
    {
        DeviceGuard guard(ctx);
        std::lock_guard<std::mutex> serial(ctx->lock);
        code = prepare(b, refs, ref_lens, qrys, qry_lens);
    }
    if (code) {
        {
            DeviceGuard guard(ctx);
            delete b;
        }
        return fail(code);
    }
    if (status) *status = 0;
    return b;
}

}  // namespace

// ------------------------------------------------------------------ the C ABI

extern "C" {

dinara_scoring_batch *dinara_scoring_batch_new(int64_t gpu, int64_t kind, int64_t pairs,
                                               const char *const *references, const int64_t *reference_lengths,
                                               const char *const *queries, const int64_t *query_lengths,
                                               const dinara_scoring *scoring, const dinara_mode *mode, int64_t eqx,
                                               int64_t threads, int64_t *status) {
    return batch_new(gpu, kind, pairs, references, reference_lengths, queries, query_lengths, scoring, mode, eqx,
                     threads, status);
}

int64_t dinara_scoring_batch_run(dinara_scoring_batch *b) {
    if (!b) return DINARA_INVALID_MODE;
    return run(b);
}

int64_t dinara_scoring_batch_scores(dinara_scoring_batch *b, int64_t *scores) {
    if (!b || !b->ran) return DINARA_INVALID_MODE;
    {
        DeviceGuard guard(b->ctx);
        if (const int64_t code = fetch(b)) return code;
    }
    // Scores may be below zero: a pair the batch cannot score fails the call with its code, the first such pair's
    // in the batch's order, as the reference's batch raises the first pair's error (api.mojo:821-841).
    for (int64_t i = 0; i < b->pairs; ++i)
        if (b->code[i] < 0) return b->code[i];
    for (int64_t i = 0; i < b->pairs; ++i) scores[i] = b->host_score[i];
    for (size_t s = 0; s < b->slot_pair.size(); ++s) scores[b->slot_pair[s]] = b->score_h[s];
    return 0;
}

// Alignments in the caller's order; `references`/`queries` must be the batch's own letters (for local spans).
int64_t dinara_scoring_batch_alignments(dinara_scoring_batch *b, const char *const *references,
                                        const char *const *queries, dinara_alignment *alignments,
                                        int64_t *statuses) {
    if (!b || !b->ran || b->kind != DINARA_BATCH_ALIGNMENTS) return DINARA_INVALID_MODE;
    {
        DeviceGuard guard(b->ctx);
        if (const int64_t code = fetch(b)) return code;
    }
    std::vector<int32_t> slot_of(b->pairs, -1);
    for (size_t s = 0; s < b->slot_pair.size(); ++s) slot_of[b->slot_pair[s]] = (int32_t)s;
    std::atomic<bool> oom{false};
    parallel_for(b->pairs, b->threads, [&](int64_t lo, int64_t hi) {
        for (int64_t p = lo; p < hi; ++p) {
            dinara_alignment &out = alignments[p];
            out.cigar = nullptr;
            out.cigar_length = 0;
            const int64_t n = b->rows[p], m = b->cols[p];
            if (b->code[p] < 0) {
                statuses[p] = b->code[p];
                continue;
            }
            int64_t score, rs = 0, re = n, qs = 0, qe = m, length = 0;
            const char *text = nullptr;
            std::string empty_side;
            if (b->code[p] == 1) {
                // An empty side: global, one gap of the other's letters; local, nothing aligned.
                score = b->host_score[p];
                if (b->local) {
                    re = qe = 0;
                } else if (n + m > 0) {
                    empty_side = std::to_string(n + m) + (n > 0 ? "D" : "I");
                    text = empty_side.data();
                    length = (int64_t)empty_side.size();
                }
            } else {
                const int32_t s = slot_of[p];
                const int32_t *v = &b->view_h[4 * s];
                score = b->score_h[s];
                if (b->local) {
                    if (v[1] == 0 && v[3] == 0) {
                        score = 0;
                        re = qe = 0;
                    } else {
                        // A local alignment's spans: the last place its letters occur (reference
                        // scoring.mojo:724-745).
                        rs = rfind(references[p], n, references[p] + v[0], v[1]);
                        re = rs + v[1];
                        qs = rfind(queries[p], m, queries[p] + v[2], v[3]);
                        qe = qs + v[3];
                    }
                }
                if (!(b->local && v[1] == 0 && v[3] == 0)) {
                    text = b->cigars_h.data() + b->cigar_offset_h[s];
                    length = b->cigar_length_h[s];
                }
            }
            char *cigar = static_cast<char *>(std::malloc(length + 1));
            if (!cigar) {
                statuses[p] = DINARA_OUT_OF_MEMORY;
                oom.store(true);
                continue;
            }
            if (length > 0) std::memcpy(cigar, text, length);
            cigar[length] = 0;
            out.cost = -score;
            out.score = score;
            out.reference_start = rs;
            out.reference_end = re;
            out.query_start = qs;
            out.query_end = qe;
            out.cigar = cigar;
            out.cigar_length = length;
            statuses[p] = 0;
        }
    });
    return 0;
}

void dinara_scoring_batch_free(dinara_scoring_batch *b) {
    if (!b) return;
    DeviceGuard guard(b->ctx);
    delete b;
}

double dinara_scoring_batch_stat(dinara_scoring_batch *b, int64_t what) {
    if (!b) return 0;
    switch (what) {
        case 0: return b->run_ms;
        case 2: return b->launches;
        case 10: return b->pass_ms[0];
        case 11: return b->pass_ms[1];
        case 12: return b->pass_ms[2];
        case 13: return b->pass_ms[3];
        default: return 0;
    }
}

int64_t dinara_gpu_scores(int64_t gpu, int64_t pairs, const char *const *references,
                          const int64_t *reference_lengths, const char *const *queries, const int64_t *query_lengths,
                          const dinara_scoring *scoring, const dinara_mode *mode, int64_t threads, int64_t *scores) {
    int64_t status = 0;
    Batch *b = batch_new(gpu, DINARA_BATCH_DISTANCES, pairs, references, reference_lengths, queries, query_lengths,
                         scoring, mode, 1, threads, &status);
    if (!b) return status;
    int64_t code = run(b);
    if (code == 0) code = dinara_scoring_batch_scores(b, scores);
    dinara_scoring_batch_free(b);
    return code;
}

int64_t dinara_gpu_scoring_alignments(int64_t gpu, int64_t pairs, const char *const *references,
                                      const int64_t *reference_lengths, const char *const *queries,
                                      const int64_t *query_lengths, const dinara_scoring *scoring,
                                      const dinara_mode *mode, int64_t eqx, int64_t threads,
                                      dinara_alignment *alignments, int64_t *statuses) {
    int64_t status = 0;
    Batch *b = batch_new(gpu, DINARA_BATCH_ALIGNMENTS, pairs, references, reference_lengths, queries,
                         query_lengths, scoring, mode, eqx, threads, &status);
    if (!b) return status;
    int64_t code = run(b);
    if (code == 0) code = dinara_scoring_batch_alignments(b, references, queries, alignments, statuses);
    dinara_scoring_batch_free(b);
    return code;
}

}  // extern "C"
