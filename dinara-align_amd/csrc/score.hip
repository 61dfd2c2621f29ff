// Gotoh's recurrence under a substitution table (Scoring), a wave or a quarter of one a pair, on MI355X (gfx950).
//
// Scores are maximized (reference gotoh.mojo:265-352): D(r, c) = max(H(r-1, c) + open, D(r-1, c) + extend),
// I(r, c) = max(H(r, c-1) + open, I(r, c-1) + extend), H(r, c) = max(H(r-1, c-1) + table[a][b], D, I), a local
// alignment floored at zero. `open` scores a gap's first letter, `extend` each later one.
//
// Layout. A pair's lanes sweep a strip of lanes * C columns, lane j holding columns jC + 1 .. jC + C, one row behind
// the lane to its left: at step s lane j takes row s - j. The cell left of a lane's first column is the left lane's
// last, of the same row, which that lane made the step before; one DPP shift hands it over, and the cell above-left
// is what came over the step before. Columns past a strip are swept strip after strip, the last column of each kept
// for the next. The table is staged in LDS as a query profile: for every letter a and every lane its C columns'
// scores table[a][query letter], so a lane reads a row's scores with one LDS load for every four columns.
//
// What bounds it is the vector unit: a cell is a sum, two maxima and a three-way maximum and the sum its right and
// lower neighbours both open a gap from, and every step pays two DPP shifts, the next row's loads and the loop besides.
// So steps inside the matrix check nothing (only a strip's first and last lanes - 1 steps do), extensions cost
// nothing where the table allows it (SH: scores held less `extend` for every row and column, a letter's score raised
// by two of them, as the borders' gaps become one constant), and pairs of up to 256 columns take 16 lanes, four pairs
// a wave: a step's own work is shared by four times the columns, and a pair of 148 letters has 15 steps of lanes
// coming in and going out rather than 63. 100,000 pairs of 148 letters: 1.72 -> 0.48 ms (4.6 T cells/s, 63 vector
// instructions for the 10 cells of a lane's step, the vector unit's rate). 5,000 queries of 300 residues in windows of
// 3,000: local ends 3.46 -> 1.63 ms (58 for 5 cells, two of them a cell the best's key), reaches 0.83 -> 0.34, spans'
// decisions 1.26 -> 0.32.
//
// Modes. SCORE_GLOBAL: H(rows, cols). SCORE_LOCAL: the best cell, above zero, by the host's rule (reference
// scored.mojo:81-84): the highest score, then the furthest along both sequences, then along the reference.
// SCORE_REACH (reference vector_score.mojo:37-162): over both prefixes reversed from a local end, the global score
// anchored there; the first cell, by anti-diagonal and then by row, that reaches the target, with the sweep cut
// off once no cell left can come earlier. SCORE_TRACE: H(rows, cols) and every cell's decision (reference
// gotoh.mojo:129-192): bit 3 a gap layer beats the aligned (on a tie the aligned comes first), bit 2 the insertion
// layer beats the deletion, bit 1 the deletion extends into the cell, bit 0 the insertion does (each only when
// strictly better than opening). A cell's bits are the signs of four differences, shifted into the word one by one; a
// wave's words are stored step by step, 256 bytes together. score_walk then walks them back as the reference's
// reconstruct does (gotoh.mojo:355-442).

#include <type_traits>

#include "cigar.h"
#include "score.h"

namespace dinara {

// Lane j of a pair reads lane j - 1's `v`; its lane 0 keeps `old`. wave_shr:1 over a wave, row_shr:1 over 16 lanes.
template <int LANES>
__device__ __forceinline__ int from_left_lane(int old, int v) {
    static_assert(LANES == 64 || LANES == 16, "a DPP row is 16 lanes");
    return __builtin_amdgcn_update_dpp(old, v, LANES == 64 ? 0x138 : 0x111, 0xF, 0xF, false);
}

// Whether (h, r, c) beats (bh, br, bc) as a local end: higher, then further along both, then along the reference.
__device__ __forceinline__ bool better_end(int h, int r, int c, int bh, int br, int bc) {
    if (h != bh) return h > bh;
    if (r + c != br + bc) return r + c > br + bc;
    return r > br;
}

// Whether (r, c) comes before (br, bc) as a reach's start: an earlier anti-diagonal, then an earlier row.
__device__ __forceinline__ bool earlier_start(int r, int c, int br, int bc) {
    if (r + c != br + bc) return r + c < br + bc;
    return r < br;
}

// A lane's scores for one letter, of the profile in LDS.
template <int C>
struct Scores {
    static constexpr int WORDS = C / 4, TAIL = score_tail(C);
    uint32_t w[(C + 3) / 4];

    __device__ __forceinline__ void load(const uint32_t *words, const uint8_t *tail, uint32_t letter) {
        const int lane = threadIdx.x;
#pragma unroll
        for (int k = 0; k < WORDS; ++k) w[k] = words[(letter * WORDS + k) * 64 + lane];
        if constexpr (TAIL == 1) w[WORDS] = tail[letter * 64 + lane];
        if constexpr (TAIL == 2) w[WORDS] = reinterpret_cast<const uint16_t *>(tail)[letter * 64 + lane];
        if constexpr (TAIL == 4) w[WORDS] = reinterpret_cast<const uint32_t *>(tail)[letter * 64 + lane];
    }
    __device__ __forceinline__ int at(int i) const { return (int)(int8_t)(w[i >> 2] >> (8 * (i & 3))); }
};

// One wave: a pair, or four of up to 256 columns. KEYED (SCORE_LOCAL): a column's best is one unsigned key,
// score << end_bits | row, so one max a cell keeps the highest score and, among equal scores, the latest row, as the
// compare-and-select form does (the host picks it where every score and row fit the key).
template <int C, int LANES, int MODE, bool SH, bool KEYED>
__device__ __forceinline__ void sweep_pairs(const ScoreArgs &a, uint8_t *lds, int slot, int rows, int cols) {
    constexpr bool LOCAL = MODE == SCORE_LOCAL;
    constexpr bool REACH = MODE == SCORE_REACH;
    constexpr bool TRACE = MODE == SCORE_TRACE;
    constexpr int PAIRS = 64 / LANES;
    constexpr int CODE_WORDS = (C + 7) / 8;
    constexpr int STRIP = LANES * C;
    const int lane = threadIdx.x & (LANES - 1);
    const int group = threadIdx.x / LANES;
    const bool valid = slot >= 0;
    const uint8_t *ref_codes = nullptr, *qry_codes = nullptr;
    if (valid) {
        const int32_t *view = a.view + 4 * (size_t)slot;
        ref_codes = a.codes + a.ref_at[slot] + view[0];
        qry_codes = a.codes + a.qry_at[slot] + view[2];
    }
    // The wave's rows: the most of its pairs, and the fewest, up to which every lane's row lies in its pair.
    int most = rows, fewest = valid ? rows : 0x7fffffff;
    if (PAIRS > 1) {
#pragma unroll
        for (int d = LANES; d < 64; d <<= 1) {
            most = max(most, __shfl_xor(most, d));
            fewest = min(fewest, __shfl_xor(fewest, d));
        }
        most = __builtin_amdgcn_readfirstlane(most);
        fewest = __builtin_amdgcn_readfirstlane(fewest);
    }
    uint32_t *words = reinterpret_cast<uint32_t *>(lds);
    uint8_t *tail = lds + (size_t)a.letters * 64 * 4 * Scores<C>::WORDS;
    uint8_t *ref = lds + (size_t)a.letters * 64 * score_lane_bytes(C) + (size_t)group * a.ref_room;
    // Four bytes of the reference's letters from `at` on, as the views read them (zero past the end).
    auto letters4 = [&](int at) {
        uint32_t w = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (at + t < rows) w |= (uint32_t)(a.reversed ? ref_codes[rows - 1 - at - t] : ref_codes[at + t]) << (8 * t);
        return w;
    };
    // A reference too long for its room goes through a ring of SCORE_RING_CHUNKS chunks instead of being staged whole.
    const bool ring = LANES == 64 && rows + 4 > a.ref_room;
    const int ref_mask = ring ? SCORE_RING - 1 : 0x7fffffff;
    if (!ring)
        for (int i = lane; i < a.ref_room; i += LANES)
            ref[i] = i < rows ? (a.reversed ? ref_codes[rows - 1 - i] : ref_codes[i]) : 0;

    const int open = SH ? a.open - a.extend : a.open, extend = SH ? 0 : a.extend;
    const int bump = SH ? -2 * a.extend : 0;   // what a letter's score is raised by
    const int rise = SH ? -a.extend : 0;       // what a held score stands above its own, a row and a column
    const int target = REACH && valid ? a.target[slot] : 0;
    const int strips = PAIRS > 1 ? 1 : (cols + STRIP - 1) / STRIP;
    int32_t *carry = strips > 1 ? a.carry + a.carry_at[blockIdx.x] : nullptr;
    uint32_t *decisions = TRACE ? a.arena + a.arena_at[blockIdx.x] : nullptr;
    const int steps = most + LANES - 1;
    // Row 0 and column 0, `letters` from the corner.
    auto border = [&](int letters) {
        return LOCAL || letters <= 0 ? 0 : SH ? open : a.open + (letters - 1) * a.extend;
    };

    int best_h = 0, best_r = 0, best_c = 0;  // SCORE_LOCAL: this lane's best end so far
    int first_r = 0, first_c = 0;            // SCORE_REACH: this lane's earliest start so far (0: none)
    int cutoff = 0x7fffffff;                 // SCORE_REACH: the wave's earliest start's anti-diagonal
    int Hp[C], Ho[C], Dp[C];                 // the row above, the lane's columns: H, H and a gap's opening, D

    for (int strip = 0; strip < strips; ++strip) {
        // A later strip's columns all lie past the earliest start found: none of them can come before it.
        if (REACH && cutoff < strip * STRIP + 2) break;
        const int c0 = strip * STRIP + lane * C;  // the column left of the lane's first
        __syncthreads();
        {
            uint32_t q[C];
#pragma unroll
            for (int i = 0; i < C; ++i) {
                const int col = c0 + i + 1;
                q[i] = col <= cols ? (a.reversed ? qry_codes[cols - col] : qry_codes[col - 1]) : 0xFFu;
            }
#pragma unroll 1
            for (int letter = 0; letter < a.letters; ++letter) {
                uint32_t w[(C + 3) / 4] = {};
#pragma unroll
                for (int i = 0; i < C; ++i) {
                    const int score = q[i] == 0xFFu ? -128 : a.table[letter * 32 + q[i]] + bump;
                    w[i >> 2] |= (uint32_t)(uint8_t)score << (8 * (i & 3));
                }
#pragma unroll
                for (int k = 0; k < Scores<C>::WORDS; ++k) words[(letter * Scores<C>::WORDS + k) * 64 + threadIdx.x] = w[k];
                constexpr int LAST = (C - 1) / 4;
                if constexpr (Scores<C>::TAIL == 1) tail[letter * 64 + threadIdx.x] = (uint8_t)w[LAST];
                if constexpr (Scores<C>::TAIL == 2)
                    reinterpret_cast<uint16_t *>(tail)[letter * 64 + threadIdx.x] = (uint16_t)w[LAST];
                if constexpr (Scores<C>::TAIL == 4) reinterpret_cast<uint32_t *>(tail)[letter * 64 + threadIdx.x] = w[LAST];
            }
        }
        // Ring: chunk k of the letters (SCORE_RING_CHUNK of them from k * SCORE_RING_CHUNK) sits in ring place
        // k mod SCORE_RING_CHUNKS. Step s reads letters s - 62 .. s + 1, so while steps 256k + 1 .. 256k + 256 run
        // chunks k - 1, k and k + 1 are held; chunk k + 1 is written at step 256k + 1, from a register loaded a
        // range of steps before, and chunk k + 2 loaded into that register.
        uint32_t pending = 0;
        if (ring) {
            static_assert(SCORE_RING_CHUNK == 4 * 64, "a chunk is four letters a lane");
            reinterpret_cast<uint32_t *>(ref)[lane] = letters4(4 * lane);
            reinterpret_cast<uint32_t *>(ref)[64 + lane] = letters4(SCORE_RING_CHUNK + 4 * lane);
            pending = letters4(2 * SCORE_RING_CHUNK + 4 * lane);
        }
        __syncthreads();

#pragma unroll
        for (int i = 0; i < C; ++i) {
            Hp[i] = border(c0 + i + 1);
            Ho[i] = Hp[i] + open;
            Dp[i] = SCORE_NEG;
        }
        int left_prev = border(c0);                // H(r - 1, c0), the cell above-left of the first column
        int out_h = SCORE_NEG, out_i = SCORE_NEG;  // H and I of the lane's last column, the row just made
        int col_h[C], col_r[C];                    // SCORE_LOCAL: per column the best
#pragma unroll
        for (int i = 0; i < C; ++i) col_h[i] = col_r[i] = 0;
        uint32_t *line = TRACE ? decisions + (size_t)strip * steps * CODE_WORDS * 64 + threadIdx.x : nullptr;

        // The row's letter is read two steps ahead, its scores one; the letter past the end is 0.
        auto letter_at = [&](int row) { return (uint32_t)ref[(min(max(row, 1), rows + 1) - 1) & ref_mask]; };
        Scores<C> prof;
        prof.load(words, tail, letter_at(1 - lane));
        uint32_t letter = letter_at(2 - lane);
        // Of several strips, the left border: rows 64k + 1 .. 64k + 64 in the lanes, the next 64 loaded.
        int kept_h = 0, kept_i = 0, next_h = 0, next_i = 0;
        auto kept = [&](int row, int &h, int &i) {
            h = border(row);
            i = SCORE_NEG;
            if (strip > 0 && row <= rows) {
                h = carry[2 * row];
                i = carry[2 * row + 1];
            }
        };
        if (LANES == 64 && strips > 1) kept(lane + 1, next_h, next_i);

        auto step = [&](int s, auto edge, auto several) {
            constexpr bool EDGE = decltype(edge)::value, SEVERAL = decltype(several)::value;
            const int r = s - lane;
            int border_h = border(s), border_i = SCORE_NEG;  // lane 0's row is s
            if (SEVERAL) {
                border_h = __builtin_amdgcn_readlane(kept_h, (s - 1) & 63);
                border_i = __builtin_amdgcn_readlane(kept_i, (s - 1) & 63);
            }
            const int lh = from_left_lane<LANES>(border_h, out_h), li = from_left_lane<LANES>(border_i, out_i);
            Scores<C> next;
            next.load(words, tail, letter);
            letter = EDGE ? letter_at(r + 2) : ref[(r + 1) & ref_mask];
            int peak = SCORE_NEG;
            if (!EDGE || (r >= 1 && r <= rows)) {
                uint32_t code[CODE_WORDS] = {};
                int ho = lh + open, il = li, h = 0;
                int sub[C];  // made before the row above is written over
#pragma unroll
                for (int i = 0; i < C; ++i) sub[i] = (i > 0 ? Hp[i - 1] : left_prev) + prof.at(i);
#pragma unroll
                for (int i = 0; i < C; ++i) {
                    const int du = Dp[i] + extend, ie = il + extend;
                    int d = max(Ho[i], du);
                    // A local end's floor: a deletion held at zero or above floors the cell as well, and one that was
                    // floored makes nothing above zero.
                    if (LOCAL) d = max(d, 0);
                    const int ins = max(ho, ie);
                    if (TRACE) {
                        const int gap = max(d, ins);
                        uint32_t &word = code[i >> 3];
                        word = __builtin_amdgcn_alignbit(word, (uint32_t)(sub[i] - gap), 31);
                        word = __builtin_amdgcn_alignbit(word, (uint32_t)(d - ins), 31);
                        word = __builtin_amdgcn_alignbit(word, (uint32_t)(Ho[i] - du), 31);
                        word = __builtin_amdgcn_alignbit(word, (uint32_t)(ho - ie), 31);
                        h = max(sub[i], gap);
                    } else {
                        h = max(max(sub[i], d), ins);
                    }
                    if constexpr (LOCAL && KEYED) {
                        col_h[i] = (int)max((uint32_t)col_h[i], ((uint32_t)h << a.end_bits) | (uint32_t)r);
                    } else if (LOCAL && h >= col_h[i] && h > 0) {
                        col_h[i] = h;
                        col_r[i] = r;
                    }
                    if (REACH) peak = max(peak, h - rise * i);
                    il = ins;
                    ho = h + open;
                    Hp[i] = h;
                    Ho[i] = ho;
                    Dp[i] = d;
                }
                out_h = h;
                out_i = il;
                left_prev = lh;
                if (SEVERAL && lane == 63) {
                    carry[2 * r] = out_h;
                    carry[2 * r + 1] = out_i;
                }
                if (TRACE) {
#pragma unroll
                    for (int k = 0; k < CODE_WORDS; ++k) line[((size_t)(s - 1) * CODE_WORDS + k) * 64] = code[k];
                }
            }
            prof = next;
            if (REACH && __any(peak >= target + rise * (r + c0 + 1))) {
                // Columns past the query's end are swept too and may reach the target: they are no start.
                if (!EDGE || (r >= 1 && r <= rows)) {
#pragma unroll
                    for (int i = 0; i < C; ++i) {
                        const int col = c0 + i + 1;
                        if (Hp[i] >= target + rise * (r + col) && col <= cols &&
                            (first_r == 0 || earlier_start(r, col, first_r, first_c))) {
                            first_r = r;
                            first_c = col;
                        }
                    }
                }
            }
        };
        // Ranges of steps between what happens now and then: the ring's refill, the kept column's next rows, and
        // SCORE_REACH's look at what the wave has found; edge steps where a lane's row can lie outside its pair.
        constexpr std::integral_constant<bool, true> yes;
        constexpr std::integral_constant<bool, false> no;
        const int range = REACH ? 32 : LANES == 64 && strips > 1 ? 64 : ring ? SCORE_RING_CHUNK : 0x40000000;
        for (int s = 1; s <= steps;) {
            if (ring && (s & (SCORE_RING_CHUNK - 1)) == 1 && s > 1) {
                const int k = s / SCORE_RING_CHUNK;
                reinterpret_cast<uint32_t *>(ref)[((k + 1) & (SCORE_RING_CHUNKS - 1)) * 64 + lane] = pending;
                pending = letters4((k + 2) * SCORE_RING_CHUNK + 4 * lane);
                __syncthreads();
            }
            if (LANES == 64 && strips > 1 && (s & 63) == 1) {
                kept_h = next_h;
                kept_i = next_i;
                kept(s + 64 + lane, next_h, next_i);
            }
            const int range_end = min(steps, ((s - 1) | (range - 1)) + 1);
            while (s <= range_end) {
                const int stop = min(range_end, s < LANES ? LANES - 1 : s <= fewest ? fewest : steps);
                const bool inside = s >= LANES && s <= fewest;
                if (LANES == 64 && strips > 1) {
                    if (inside)
                        for (; s <= stop; ++s) step(s, no, yes);
                    else
                        for (; s <= stop; ++s) step(s, yes, yes);
                } else {
                    if (inside)
                        for (; s <= stop; ++s) step(s, no, no);
                    else
                        for (; s <= stop; ++s) step(s, yes, no);
                }
            }
            if (REACH && __any(first_r != 0)) {
                // Every cell still to come lies on anti-diagonal s + 1 or later (s the next step), so an earliest
                // start before that is final.
                int diag = first_r != 0 ? first_r + first_c : 0x7fffffff;
#pragma unroll
                for (int d = 1; d < 64; d <<= 1) diag = min(diag, __shfl_xor(diag, d));
                cutoff = diag;
                if (diag < s + 1) break;
            }
        }
        // Fold the strip's columns into the lane's own candidate.
        if (LOCAL) {
#pragma unroll
            for (int i = 0; i < C; ++i) {
                const int col = c0 + i + 1;
                if (col > cols) continue;
                if (KEYED) {
                    col_r[i] = (int)((uint32_t)col_h[i] & ((1u << a.end_bits) - 1u));
                    col_h[i] = (int)((uint32_t)col_h[i] >> a.end_bits);
                }
                if (col_h[i] > 0 && better_end(col_h[i], col_r[i], col, best_h, best_r, best_c)) {
                    best_h = col_h[i];
                    best_r = col_r[i];
                    best_c = col;
                }
            }
        }
        if (carry) __threadfence_block();
    }

    if ((MODE == SCORE_GLOBAL || TRACE) && valid) {
        // The last strip's rows end at the pair's last: the lane of its last column holds the corner.
        const int last = cols - 1 - (strips - 1) * STRIP;
        if (lane == last / C) {
            int corner = Hp[0];
#pragma unroll
            for (int i = 1; i < C; ++i) corner = last % C == i ? Hp[i] : corner;
            a.score[slot] = corner - rise * (rows + cols);
        }
        if (TRACE && lane == 0) {
            a.walk_base[slot] = reinterpret_cast<uint64_t>(decisions + group * LANES);
            a.walk_columns[slot] = C;
        }
    }
    if (LOCAL) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int oh = __shfl_xor(best_h, d), orow = __shfl_xor(best_r, d), ocol = __shfl_xor(best_c, d);
            if (oh > 0 && (best_h == 0 || better_end(oh, orow, ocol, best_h, best_r, best_c))) {
                best_h = oh;
                best_r = orow;
                best_c = ocol;
            }
        }
        if (lane == 0) {
            a.score[slot] = best_h;
            a.end_row[slot] = best_r;
            a.end_col[slot] = best_c;
        }
    }
    if (REACH) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int orow = __shfl_xor(first_r, d), ocol = __shfl_xor(first_c, d);
            if (orow != 0 && (first_r == 0 || earlier_start(orow, ocol, first_r, first_c))) {
                first_r = orow;
                first_c = ocol;
            }
        }
        if (lane == 0) {
            a.end_row[slot] = first_r;
            a.end_col[slot] = first_c;
        }
    }
}

// One launch for a pass's pairs of one kind, each wave taking the columns a lane that its own pairs need.
template <int LANES, int MODE, bool SH, bool KEYED = false>
__global__ __launch_bounds__(64) void score_wave(ScoreArgs a) {
    extern __shared__ uint8_t lds[];
    const int index = blockIdx.x * (64 / LANES) + threadIdx.x / LANES;
    int slot = -1, rows = 0, cols = 0;
    if (index < a.count) {
        slot = a.list[index];
        rows = a.view[4 * (size_t)slot + 1];
        cols = a.view[4 * (size_t)slot + 3];
    }
    int widest = cols;
#pragma unroll
    for (int d = LANES; d < 64; d <<= 1) widest = max(widest, __shfl_xor(widest, d));
    if (LANES == 64) {
        slot = __builtin_amdgcn_readfirstlane(slot);
        rows = __builtin_amdgcn_readfirstlane(rows);
        cols = __builtin_amdgcn_readfirstlane(cols);
    }
#define SCORE_COLUMNS(C) \
    case C: sweep_pairs<C, LANES, MODE, SH, KEYED>(a, lds, slot, rows, cols); break;
    switch (score_columns(LANES, __builtin_amdgcn_readfirstlane(widest))) {
        SCORE_COLUMNS(1)
        SCORE_COLUMNS(2)
        SCORE_COLUMNS(3)
        SCORE_COLUMNS(4)
        SCORE_COLUMNS(5)
        SCORE_COLUMNS(6)
        SCORE_COLUMNS(7)
        SCORE_COLUMNS(8)
    }
    if constexpr (LANES == SCORE_NARROW) {
        switch (score_columns(LANES, __builtin_amdgcn_readfirstlane(widest))) {
            SCORE_COLUMNS(9)
            SCORE_COLUMNS(10)
            SCORE_COLUMNS(11)
            SCORE_COLUMNS(12)
            SCORE_COLUMNS(13)
            SCORE_COLUMNS(14)
            SCORE_COLUMNS(15)
            SCORE_COLUMNS(16)
        }
    }
#undef SCORE_COLUMNS
}

// The walk back through SCORE_TRACE's decisions, 16 lanes a pair (reference gotoh.mojo:355-442): from the aligned
// layer follow the source; a gap layer keeps stepping while the cell says it extends; at row 0 or column 0 the rest is
// gaps. A move's decision is known only once the move before it is made, so what bounds a walk is one load after
// another: the lanes read the next 16 cells along the way the walk is going (the diagonal, or the gap's row or column)
// at once, and take all the moves up to where it turns. 5,000 walks over 300 residues at 30% differences: 0.70 ms with
// a thread a pair and a load a move, 0.27 so. Then every pair's CIGAR goes into the shared output.
__global__ __launch_bounds__(256) void score_walk(ScoreArgs a) {
    const int lane = threadIdx.x & 15;
    const int shift = threadIdx.x & 48;  // the pair's lanes within its wave
    const int index = blockIdx.x * 16 + threadIdx.x / 16;
    int64_t moves = -1;
    int slot = 0;
    if (index < a.count) {
        slot = a.list[index];
        const int32_t *view = a.view + 4 * (size_t)slot;
        const int rows = view[1], cols = view[3];
        const uint8_t *ref = a.codes + a.ref_at[slot] + view[0];
        const uint8_t *qry = a.codes + a.qry_at[slot] + view[2];
        const uint32_t *decisions = reinterpret_cast<const uint32_t *>(a.walk_base[slot]);
        const int columns = a.walk_columns[slot], words = (columns + 7) >> 3;
        const int strip_cols = a.lanes * columns;
        const int64_t strip_words = (int64_t)(rows + a.lanes - 1) * words * 64;  // one strip only under 64 lanes
        // Every lane of the pair holds the same tape and writes the same words.
        OpTape ops{reinterpret_cast<uint64_t *>(a.op_scratch + a.op_base[slot]), 0, 0};
        int r = rows, c = cols, layer = 0;
        while (r > 0 && c > 0) {
            const int lr = r - (layer != 2 ? lane : 0), lc = c - (layer != 1 ? lane : 0);
            const bool in = lr > 0 && lc > 0;
            uint32_t nib = 0, unequal = 0;
            if (in) {
                const int col = lc - 1, strip = col / strip_cols, within = col - strip * strip_cols;
                const int at = within / columns, cell = within - at * columns;
                const int last = min(columns - (cell & 8), 8) - 1;  // the word's first cell is its highest nibble
                const uint32_t word =
                    decisions[strip * strip_words + ((int64_t)(lr + at - 1) * words + (cell >> 3)) * 64 + at];
                nib = (word >> (4 * (last - (cell & 7)))) & 15u;
                if (layer == 0) unequal = a.eqx && ref[lr - 1] != qry[lc - 1];
            }
            // The lanes, from 0 on, whose move goes on the way the walk is going.
            const bool goes = in && (layer == 0 ? !(nib & 8u) : (nib & (layer == 1 ? 2u : 1u)) != 0);
            const uint32_t stay = (uint32_t)(__ballot(goes) >> shift) & 0xFFFFu;
            int run = __builtin_ctz(~stay);
            if (layer == 0) {
                if (run > 0) {
                    uint64_t codes = (__ballot(unequal != 0) >> shift) & 0xFFFFull & ((1ull << run) - 1);
                    codes = (codes | (codes << 8)) & 0x00FF00FFull;
                    codes = (codes | (codes << 4)) & 0x0F0F0F0Full;
                    codes = (codes | (codes << 2)) & 0x33333333ull;
                    codes = (codes | (codes << 1)) & 0x55555555ull;
                    ops.put_many(codes, run);
                    r -= run;
                    c -= run;
                }
                if (run < 16 && r > 0 && c > 0) {
                    // This cell comes from a gap: its first move here, and whether the gap goes on.
                    const uint32_t turn = __shfl((int)nib, shift + run);
                    const int from = (turn & 4u) ? 2 : 1;
                    ops.put((uint32_t)from + 1);
                    if (from == 1) --r;
                    else --c;
                    layer = (turn & (from == 1 ? 2u : 1u)) ? from : 0;
                }
            } else {
                // Moves of the gap's layer: `run` cells that extend, then the one it opened from, if it lies in the
                // matrix and among the lanes.
                const int left = layer == 1 ? r : c;
                const bool opened = run < 16 && run < left;
                const int count = opened ? run + 1 : run;
                ops.put_many(0x5555555555555555ull * (uint64_t)(layer + 1) & ((1ull << (2 * count)) - 1), count);
                if (layer == 1) r -= count;
                else c -= count;
                if (opened) layer = 0;
            }
        }
        for (; r > 0; --r) ops.put(2u);
        for (; c > 0; --c) ops.put(3u);
        ops.close();
        if (lane == 0) moves = ops.count;
    }
    const uint64_t *words = reinterpret_cast<const uint64_t *>(a.op_scratch + (moves >= 0 ? a.op_base[slot] : 0));
    publish_wave(a.eqx, 0, words, moves, a.cigars, a.cigar_used, a.cigar_offset + slot, a.cigar_length + slot);
}

// ------------------------------------------------------------------ launches

template <int LANES, int MODE>
static void launch_mode(const ScoreArgs &a, dim3 grid, size_t lds, hipStream_t stream) {
    if (a.shifted) hipLaunchKernelGGL((score_wave<LANES, MODE, true>), grid, dim3(64), lds, stream, a);
    else if constexpr (LANES == 64)
        hipLaunchKernelGGL((score_wave<LANES, MODE, false>), grid, dim3(64), lds, stream, a);
}

void launch_score(const ScoreArgs &a, size_t lds, hipStream_t stream) {
    if (a.count <= 0) return;
    const int pairs = 64 / a.lanes;
    const dim3 grid((a.count + pairs - 1) / pairs), block(64);
    switch (a.mode) {
        case SCORE_GLOBAL:
            if (a.lanes == SCORE_NARROW) launch_mode<SCORE_NARROW, SCORE_GLOBAL>(a, grid, lds, stream);
            else launch_mode<64, SCORE_GLOBAL>(a, grid, lds, stream);
            break;
        case SCORE_LOCAL:
            if (a.end_bits > 0) hipLaunchKernelGGL((score_wave<64, SCORE_LOCAL, false, true>), grid, block, lds, stream, a);
            else hipLaunchKernelGGL((score_wave<64, SCORE_LOCAL, false, false>), grid, block, lds, stream, a);
            break;
        case SCORE_REACH: launch_mode<64, SCORE_REACH>(a, grid, lds, stream); break;
        default:
            if (a.lanes == SCORE_NARROW) launch_mode<SCORE_NARROW, SCORE_TRACE>(a, grid, lds, stream);
            else launch_mode<64, SCORE_TRACE>(a, grid, lds, stream);
            break;
    }
}

void launch_score_walk(const ScoreArgs &a, hipStream_t stream) {
    if (a.count <= 0) return;
    hipLaunchKernelGGL(score_walk, dim3((a.count + 15) / 16), dim3(256), 0, stream, a);
}

}  // namespace dinara
