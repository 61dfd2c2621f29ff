// The strip sweep on MI355X (gfx950): Gotoh's recurrence in cost form over a band of diagonals (or the whole matrix),
// each cell's decision kept under the reference's flag rule, then the walk back (reference lanes.mojo:795-947
// recurrence, :905-923 flags, :1410-1460 walk). It takes the bands too wide for a group of sixteen lanes, two-piece
// gaps and free ends but for short pairs in narrow bands (sweep.hip), and the pairs no band settles.
//
// Layout. The query's columns are cut into strips of 64 C (C = 2, 4 or 8 a lane); a wave sweeps a strip top to bottom
// over the rows whose cells there hold the band, lane j holding columns c0 + 1 .. c0 + C (c0 = strip * 64 C + jC) one
// row behind lane j - 1: at step s lane j takes the strip's row s - j. A cell's left neighbours come from the lane to
// the left, made the step before, by one DPP wave_shr:1; the cells above are the lane's own registers. What lies
// outside the strip's rows is unreachable: above its first row every diagonal is past the band's highest, and left of
// its rows past the left strip's last every diagonal is below its lowest, so every path inside the band is swept, and
// paths a little outside it: the cost found is no more than the band's least, and the certificate holds for it.
//
// A strip's lane 0 takes its left neighbours from the last column of the strip to its left, which that strip's lane 63
// writes to a carry record a row, with a relaxed agent-scope atomic store: the record's own nonzero value says it is
// there, so no fence or flag is needed, and agent scope keeps it coherent across the XCDs' L2s. The reading wave
// fetches 64 rows' records at once (lane i row s + i) every 64 steps, and lane 0 takes row s's with a readlane; column
// 0's borders are made the same way. So a pair's strips run as a pipeline over the whole chip, each 64 C + 128 rows or
// so behind the one to its left, and one launch takes every pair of a round, whatever its band, or as many of them as
// its decisions and carry records find room for. Waves claim strips in the host's order, in which a strip always
// follows the one to its left (which is then held by a running wave), the pairs with the most strips first (their
// pipelines are the launch's longest chains); every wait gives up after STRIP_POLL_LIMIT polls, and the host sweeps the
// pairs that leaves unsettled whole.
//
// The reference's letters pass through a ring in LDS, 64 written every 64 steps and loaded 64 steps before that; the
// lane's query letters sit in registers. Between refills a step is the cells, two DPP moves, the letter's read and the
// stores: a pair of 20,000 letters is a chain of 25,000 steps, whose every instruction counts.
// Checks and refills at every step instead: 360 ns a step of eight columns a lane, 198 so (2,000 uneven gap-affine
// distances 19.5 -> 14.5 ms, 1,000 two-piece CIGARs 14.5 -> 11.5, 5,000 reads in windows 3.95 -> 3.3).
//
// One gap piece (ONE): values and decisions as the group sweep's (group.hip): with decisions kept, cost * 16 + a tag
// whose minimum breaks ties the reference's way, a cell's nibble bits 3:2 (source + 3) mod 4 (source 0 two unequal
// letters, 1 the deletion layer, 2 the insertion layer, 3 two equal), bit 1 D(r+1, c) opened, bit 0 I(r, c+1) opened.
// With both extensions equal (SH) values are held shifted, H - e(r + c), so an extension costs nothing. Two pieces: a
// byte a cell, bits 0-2 the source (0 equal, 5 unequal, 1 and 3 the pieces' deletions, 2 and 4 their insertions), bit 2
// + L layer L extends into the cell. A lane's record of a row is its C cells, low first, at the pair's first decision +
// ((strip * rows + r - the strip's first row) * 64 + lane) * strip_record_bytes.

#include <type_traits>

#include "bands.h"
#include "strip.h"

namespace dinara {

namespace {

constexpr int SEGMENT = 64;     // steps between refills: of the ring of letters, and of the left neighbours
constexpr int RING = 4 * SEGMENT;
constexpr int TAG_INF = 1 << 30;  // unreachable: above every real tagged value, with room to add

__device__ __forceinline__ int from_left_lane(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, 0x138, 0xF, 0xF, false);
}

// A gap of `letters` letters at its cheaper piece (none: nothing).
template <int P>
__device__ __forceinline__ int gap_of(int open, int ext, int open2, int ext2, int letters) {
    if (letters <= 0) return 0;
    const int one = open + letters * ext;
    return P == 2 ? min(one, open2 + letters * ext2) : one;
}

// Carry records: a value in 32 bits, never zero (every value lies above -2^30).
__device__ __forceinline__ uint32_t carried(int v) { return (uint32_t)v + 0x40000000u; }
__device__ __forceinline__ int uncarried(uint32_t v) { return (int)(v - 0x40000000u); }
__device__ __forceinline__ unsigned long long carry_record(int h, int i) {
    return ((unsigned long long)carried(h) << 32) | carried(i);
}

// The sequence letters a slot (or its view) sweeps.
struct Letters {
    const uint32_t *ref, *qry;
    int bits, shift, n, m, ref_at, qry_at;  // a tape word holds 1 << shift letters
    uint32_t mask;
    bool back;

    __device__ uint32_t at(const uint32_t *words, int x) const {
        return (words[(size_t)(x >> shift) * 64] >> (bits * (x & ((1 << shift) - 1)))) & mask;
    }
    __device__ uint32_t query(int i) const { return at(qry, back ? qry_at + m - 1 - i : qry_at + i); }
    __device__ uint32_t reference(int i) const {  // zero past the end
        return i < n ? at(ref, back ? ref_at + n - 1 - i : ref_at + i) : 0u;
    }
};

// The letters a slot (or its view) sweeps and its free ends: reference start, end, query start, end.
template <bool FREE>
struct Sides {
    int n, m, free[4];
    __device__ Sides(const SweepArgs &s, int slot) {
        n = FREE ? s.view_rows[slot] : s.tape.rows[slot];
        m = FREE ? s.view_cols[slot] : s.tape.cols[slot];
#pragma unroll
        for (int f = 0; f < 4; ++f) free[f] = FREE ? s.free[4 * slot + f] : 0;
    }
};

// What a strip leaves: in the lane that found it, the pair's cost and (free ends) the diagonal it ends on.
struct Ending {
    bool mine = false;
    int cost = 0, diagonal = 0;
};

// What a finished pair's cost settles: whole matrices every pair, bands those the certificate proves; the others are
// filed with the band their cost proves. One lane.
template <bool FREE>
__device__ __forceinline__ void finish_pair(const StripArgs &a, const StripPair &p, const StripPair *at,
                                            const Ending &end) {
    const SweepArgs &s = a.s;
    const Sides<FREE> of(s, p.slot);
    const int n = of.n, m = of.m;
    if (!a.whole) {
        int want_low = 0, want_high = 0;
        const bool proven =
            FREE ? end.cost < INF && certify_ends(s, n, m, end.cost, p.lo, p.hi, of.free, &want_low, &want_high)
                 : certify(s, n, m, end.cost, p.lo, p.hi, &want_low, &want_high);
        if (!proven) {
            if (FREE && end.cost >= INF) {  // no end in the band: the whole matrix's diagonals next
                want_low = -n;
                want_high = m;
            }
            file_retry(s, p.slot, n + m, want_low, want_high);
            return;
        }
    }
    if (FREE) {
        // The end cell on that diagonal: column m (at or above the corner's diagonal) or row n (below it).
        s.end_row[p.slot] = end.diagonal >= m - n ? m - end.diagonal : n;
        s.end_col[p.slot] = end.diagonal >= m - n ? m : n + end.diagonal;
    }
    s.cost[p.slot] = end.cost;
    s.status[p.slot] = 0;
    s.walk_class[p.slot] = CLASS_STRIP_FIRST;
    s.walk_flags[p.slot] = reinterpret_cast<uint64_t>(at);  // this launch settled it (strip_walk)
}

// An empty side: one gap of the other's letters, or under free ends the cheapest of the cells along the other side that
// may end (their costs never fall).
template <int P, bool FREE>
__device__ __forceinline__ Ending empty_side(const StripArgs &a, const Sides<FREE> &of) {
    const CostParams &k = a.s.costs;
    const int length = of.n == 0 ? of.m : of.n;
    const int start = of.free[of.n == 0 ? 2 : 0], stop = of.free[of.n == 0 ? 3 : 1];
    const int first = length - stop > 0 ? length - stop : 0;  // the cheapest end, and the last one as cheap
    const int last = first <= start ? (start < length ? start : length) : first;
    Ending end;
    end.mine = true;
    end.cost = of.n == 0 ? gap_of<P>(k.ins_open, k.ins_ext, k.ins_open2, k.ins_ext2, first - start)
                         : gap_of<P>(k.del_open, k.del_ext, k.del_open2, k.del_ext2, first - start);
    end.diagonal = of.n == 0 ? (a.s.lowest_end ? last : first) : (a.s.lowest_end ? -first : -last);
    return end;
}

// A better end than the one held: cheaper, then a higher library diagonal (a lower lane diagonal), or with
// `lowest_end` a lower one. As one key: the cost, then the diagonal's rank.
__device__ __forceinline__ unsigned long long end_key(int cost, int diagonal, int lowest_end) {
    const uint32_t rank = (uint32_t)(lowest_end ? -diagonal : diagonal) + 0x40000000u;
    return ((unsigned long long)(uint32_t)cost << 32) | rank;
}
__device__ __forceinline__ int key_diagonal(unsigned long long key, int lowest_end) {
    const int d = (int)((uint32_t)key - 0x40000000u);
    return lowest_end ? -d : d;
}

// One strip. Returns false when a wait for the left strip gave up; else leaves in `ending` what it found.
template <int C, int P, bool RECORD, bool SH, bool FREE>
__device__ __forceinline__ bool sweep_strip(const StripArgs &a, const StripPair &p, int pair, int strip,
                                            uint8_t *ring, Ending &ending) {
    constexpr bool ONE = P == 1;
    constexpr bool TAGS = ONE && RECORD;
    constexpr int SCALE = TAGS ? 16 : 1;
    constexpr int FAR = ONE ? TAG_INF : INF;  // unreachable
    const int lane = threadIdx.x;
    const CostParams k = a.s.costs;
    const int slot = p.slot;
    const Sides<FREE> of(a.s, slot);
    const int n = of.n, m = of.m;
    Letters text;
    {
        const int group = slot >> 6;
        text.ref = a.s.tape.words + a.s.tape.group_base[group] + (slot & 63);
        text.qry = text.ref + (size_t)a.s.tape.group_ref_words[group] * 64;
        text.bits = a.s.tape.bits;
        text.shift = text.bits == 2 ? 4 : 2;
        text.mask = (1u << text.bits) - 1;
        text.n = n;
        text.m = m;
        text.ref_at = FREE ? a.s.view_ref_at[slot] : 0;
        text.qry_at = FREE ? a.s.view_qry_at[slot] : 0;
        text.back = FREE && a.s.view_reversed;
    }
    if (n == 0 || m == 0) {  // one strip; the walk makes the gap
        ending = empty_side<P, FREE>(a, of);
        ending.mine = lane == 0;
        return true;
    }
    const int e = SH ? k.del_ext : 0;
    // The borders: row 0 and column 0, as values (shifted, times the tags' room).
    const auto top_border = [&](int c) {
        return (gap_of<P>(k.ins_open, k.ins_ext, k.ins_open2, k.ins_ext2, c - of.free[2]) - e * c) * SCALE;
    };
    const auto left_border = [&](int r) {
        return (gap_of<P>(k.del_open, k.del_ext, k.del_open2, k.del_ext2, r - of.free[0]) - e * r) * SCALE;
    };
    // One piece: what a cell's steps add, with their tags.
    const int sub_eq = -2 * e * SCALE + (TAGS ? 12 : 0), sub_ne = (k.mismatch - 2 * e) * SCALE;
    const int open_d = k.del_open * SCALE + (TAGS ? 6 : 0), open_i = k.ins_open * SCALE + (TAGS ? 9 : 0);
    const int ext_d = SH ? 0 : k.del_ext * SCALE, ext_i = SH ? 0 : k.ins_ext * SCALE;

    const int first = strip_first_row(p, strip), last = strip_last_row(p, strip, n);
    const int left_first = strip > 0 ? strip_first_row(p, strip - 1) : 1;
    const int left_last = strip > 0 ? strip_last_row(p, strip - 1, n) : n;
    const bool last_strip = strip + 1 == p.strips;
    const int c0 = strip * strip_columns(C) + lane * C;  // the column left of the lane's first
    uint32_t q[C];
#pragma unroll
    for (int i = 0; i < C; ++i) q[i] = c0 + i + 1 <= m ? text.query(c0 + i) : 0xFFFFu;
    // The row above: H, and D as the next row takes it (one piece: D(r + 1, c); two: D(r, c) of both pieces).
    int H[C], D[C], D2[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
        H[i] = first == 1 ? top_border(c0 + i + 1) : FAR;
        D[i] = ONE && first == 1 ? H[i] + open_d + ext_d : FAR;
        D2[i] = FAR;
    }
    int left_prev = first == 1 ? top_border(c0) : FAR;  // H(r - 1, c0)
    // The lane's last column, the row it just made: H, and I as the next column takes it.
    int out_h = FAR, out_i = FAR, out_i2 = FAR;
    unsigned long long *const carry = a.carry + p.carry_at;
    const unsigned long long *const left_carry = strip > 0 ? carry + (size_t)(strip - 1) * p.rows * P : nullptr;
    unsigned long long *const own_carry = last_strip ? nullptr : carry + (size_t)strip * p.rows * P;
    // The left neighbours of the segment's rows, lane t's that of its row t: H, and I as column c0 + 1 takes it.
    int left_h = FAR, left_i = FAR, left_i2 = FAR;
    // Those of row `row` (this lane's) from the left strip's records, waited for; unreachable where `want` is not set.
    const auto fetch = [&](int row, bool want) __attribute__((always_inline)) {
        const unsigned long long *from = left_carry + (size_t)(want ? row - left_first : 0) * P;
        unsigned long long record = 0, record2 = 0;
        for (int polls = 0;; ++polls) {
            if (want) {
                record = __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (P == 2) record2 = __hip_atomic_load(from + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            const bool missing = want && (record == 0 || (P == 2 && record2 == 0));
            if (__ballot(missing) == 0) break;
            if (polls > a.polls) return false;
            __builtin_amdgcn_s_sleep(2);
        }
        left_h = want ? uncarried((uint32_t)(record >> 32)) : FAR;
        left_i = want ? uncarried((uint32_t)record) : FAR;
        left_i2 = P == 2 && want ? uncarried((uint32_t)record2) : FAR;
        return true;
    };
    if (left_carry && first > 1) {  // the cell above-left of the strip's first: on the band's highest diagonal
        if (!fetch(first - 1, true)) return false;
        if (lane == 0) left_prev = left_h;
    }

    // The ring holds the letters of the segment's steps and the one before (row r's letter is r - 1; lane j reads letter
    // first - 1 + s - j at step s = 0, 1, ...) and the next segment's; the one after's wait in a register.
    __syncthreads();
    ring[(first - 1 + lane) & (RING - 1)] = (uint8_t)text.reference(first - 1 + lane);
    ring[(first - 1 + SEGMENT + lane) & (RING - 1)] = (uint8_t)text.reference(first - 1 + SEGMENT + lane);
    uint32_t pending = text.reference(first - 1 + 2 * SEGMENT + lane);
    __syncthreads();

    // Free ends: the least key of this lane's ends so far. Column m's lane and place, and the rows and columns that
    // may end.
    unsigned long long best = ~0ull;
    const int end_place = m - c0 - 1;  // the place of column m in this lane, when 0 .. C - 1
    const int end_row_from = n - of.free[1], end_col_from = m - of.free[3];
    const auto consider = [&](int value, int r, int c) {
        const int shift = e * (r + c) * SCALE;
        if (value >= FAR - shift) return;  // unreachable
        const unsigned long long key = end_key((value + shift) / SCALE, c - r, a.s.lowest_end);
        if (key < best) best = key;
    };
    if (FREE) {
        // The borders' own ends: row 0 in column m, column 0 in row n.
        if (end_place >= 0 && end_place < C && end_row_from <= 0) consider(top_border(m), 0, m);
        if (lane == 0 && strip == 0 && end_col_from <= 0) consider(left_border(n), n, 0);
    }
    int corner = FAR;
    // Decisions: a row's records are 64 lanes', and lane j is j rows behind lane 0: from the place of lane 63's, each
    // lane's lies a fixed way on.
    constexpr int BYTES = strip_record_bytes(C, P);
    uint8_t *record_base =
        RECORD ? a.decisions + p.decision_at + ((int64_t)strip * p.rows - 63) * (64 * BYTES) : nullptr;
    const uint32_t record_off = (uint32_t)((63 - lane) * 64 + lane) * BYTES;

    const int rows = last - first + 1, steps = rows + 63;
    uint32_t letter = ring[(first - 1 - lane) & (RING - 1)];
    // Step s (lane 0's row is first + s), t its place in the segment. EDGE: lanes may be above the strip's first row or
    // below its last, and the last row's ends are looked at.
    const auto step = [&](auto edge, int s, int t) __attribute__((always_inline)) {
        constexpr bool EDGE = edge.value;
        const uint32_t next_letter = ring[(first + s - lane) & (RING - 1)];
        const int r = first + s - lane;
        const int lh = from_left_lane(__builtin_amdgcn_readlane(left_h, t), out_h);
        const int li = from_left_lane(__builtin_amdgcn_readlane(left_i, t), out_i);
        const int li2 = P == 2 ? from_left_lane(__builtin_amdgcn_readlane(left_i2, t), out_i2) : FAR;
        if (!EDGE || (r >= first && r <= last)) {
            int hl = lh, il = li, il2 = li2, hd = left_prev;
            uint32_t nibbles = 0;
            unsigned long long bytes = 0;
#pragma unroll
            for (int i = 0; i < C; ++i) {
                const bool eq = q[i] == letter;
                const int hu = H[i];
                int h;
                if constexpr (ONE) {
                    const int sub = hd + (eq ? sub_eq : sub_ne);
                    const int dc = TAGS ? (D[i] & ~2) : D[i];
                    const int ic = TAGS ? (il & ~1) : il;
                    const int low = min(sub, min(dc, ic));
                    h = TAGS ? (low & ~15) : low;
                    const int dn = min(h + open_d, dc) + ext_d, in = min(h + open_i, ic) + ext_i;
                    if (TAGS) nibbles = __builtin_amdgcn_alignbit((uint32_t)((dn ^ in) + low), nibbles, 4);
                    D[i] = dn;
                    il = in;
                } else {
                    const int od = hu + k.del_first, ed = D[i] + k.del_ext;
                    const int oi = hl + k.ins_first, ei = il + k.ins_ext;
                    const int od2 = hu + k.del_first2, ed2 = D2[i] + k.del_ext2;
                    const int oi2 = hl + k.ins_first2, ei2 = il2 + k.ins_ext2;
                    const int d = min(od, ed), ins = min(oi, ei), d2 = min(od2, ed2), ins2 = min(oi2, ei2);
                    const int sub = hd + (eq ? 0 : k.mismatch);
                    h = min(min(sub, min(d, ins)), min(d2, ins2));
                    if (RECORD) {
                        // The lowest priority first, each later source as cheap as the cell taking over.
                        uint32_t src = eq ? 0u : 5u;
                        src = ins == h ? 2u : src;
                        src = ins2 == h ? 4u : src;
                        src = d == h ? 1u : src;
                        src = d2 == h ? 3u : src;
                        src = (!eq && sub == h) ? 5u : src;
                        const uint32_t flag = src | (ed <= od ? 8u : 0u) | (ei <= oi ? 16u : 0u) |
                                              (ed2 <= od2 ? 32u : 0u) | (ei2 <= oi2 ? 64u : 0u);
                        if (i < 4) nibbles |= flag << (8 * i);
                        else bytes |= (unsigned long long)flag << (8 * i);
                    }
                    D[i] = d;
                    D2[i] = d2;
                    il = ins;
                    il2 = ins2;
                }
                hd = hu;
                hl = h;
                H[i] = h;
            }
            out_h = hl;
            out_i = il;
            out_i2 = il2;
            left_prev = lh;
            if (RECORD) {
                uint8_t *to = record_base + record_off;
                if constexpr (ONE) {
                    if constexpr (C == 8) *reinterpret_cast<uint32_t *>(to) = nibbles;
                    else if constexpr (C == 4) *reinterpret_cast<uint16_t *>(to) = (uint16_t)(nibbles >> 16);
                    else *to = (uint8_t)(nibbles >> 24);
                } else {
                    if constexpr (C == 8) *reinterpret_cast<unsigned long long *>(to) = bytes | nibbles;
                    else if constexpr (C == 4) *reinterpret_cast<uint32_t *>(to) = nibbles;
                    else *reinterpret_cast<uint16_t *>(to) = (uint16_t)nibbles;
                }
            }
            if (own_carry && lane == 63) {
                unsigned long long *to = own_carry + (int64_t)(s - 63) * P;
                __hip_atomic_store(to, carry_record(out_h, out_i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (P == 2)
                    __hip_atomic_store(to + 1, carry_record(0, out_i2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (FREE) {
                if (last_strip && r >= end_row_from) {
                    int end = FAR;
#pragma unroll
                    for (int i = 0; i < C; ++i) end = i == end_place ? H[i] : end;
                    if (end_place >= 0 && end_place < C) consider(end, r, m);
                }
                if (EDGE && r == n) {
#pragma unroll
                    for (int i = 0; i < C; ++i)
                        if (c0 + i + 1 <= m && c0 + i + 1 >= end_col_from) consider(H[i], n, c0 + i + 1);
                }
            } else if (EDGE && last_strip && r == n) {
#pragma unroll
                for (int i = 0; i < C; ++i) corner = i == end_place ? H[i] : corner;
            }
        }
        if (RECORD) record_base += 64 * BYTES;
        letter = next_letter;
    };
    for (int s0 = 0; s0 < steps; s0 += SEGMENT) {
        if (s0 > 0) {
            ring[(first - 1 + s0 + SEGMENT + lane) & (RING - 1)] = (uint8_t)pending;
            pending = text.reference(first - 1 + s0 + 2 * SEGMENT + lane);
            __syncthreads();
        }
        const int row = first + s0 + lane;
        if (!left_carry) {
            left_h = left_border(row);
            left_i = ONE ? left_h + open_i + ext_i : FAR;
        } else if (!fetch(row, row <= left_last && row <= last)) {
            return false;
        }
        if (s0 > 0 && s0 + SEGMENT < rows) {
#pragma unroll 2
            for (int t = 0; t < SEGMENT; ++t) step(std::false_type(), s0 + t, t);
        } else {
            const int here = steps - s0 < SEGMENT ? steps - s0 : SEGMENT;
            for (int t = 0; t < here; ++t) step(std::true_type(), s0 + t, t);
        }
    }

    if (!FREE) {
        const int shift = e * (n + m) * SCALE;
        ending.mine = last_strip && end_place >= 0 && end_place < C;  // the corner's lane
        ending.cost = corner >= FAR - shift ? INF : (corner + shift) / SCALE;
        return true;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long other = __shfl_xor(best, d);
        best = other < best ? other : best;
    }
    ending.mine = lane == 0;
    if (p.strips > 1 && lane == 0) {
        // The least over the strips: each returns before its strip is counted, so the last to be counted finds them
        // all.
        const unsigned long long before =
            __hip_atomic_fetch_min(&a.best[pair], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int counted = before == 0 ? 2 : 1;  // takes the returned value; no key is 0, so 1
        ending.mine = __hip_atomic_fetch_add(&a.done[pair], counted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
                      p.strips;
        if (ending.mine) best = __hip_atomic_load(&a.best[pair], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    ending.cost = best == ~0ull ? INF : (int)(best >> 32);
    ending.diagonal = best == ~0ull ? 0 : key_diagonal(best, a.s.lowest_end);
    return true;
}

template <int P, bool RECORD, bool SH, bool FREE>
__global__ __launch_bounds__(64) void strip_sweep(StripArgs a) {
    __shared__ uint8_t ring[RING];
    for (;;) {
        // The wave comes together before it claims. Without this the compiler joined "lane 0 settles the pair", at a
        // strip's end, to "lane 0 claims", here, and sent the other lanes round again without lane 0, to sweep strip 0
        // for ever.
        __syncthreads();
        int claimed = 0;
        if (threadIdx.x == 0) claimed = atomicAdd(a.claim, 1);
        claimed = __builtin_amdgcn_readfirstlane(claimed);
        if (claimed >= a.strips) return;
        const int2 which = a.order ? a.order[claimed] : make_int2(claimed, 0);
        const int pair = __builtin_amdgcn_readfirstlane(which.x), strip = __builtin_amdgcn_readfirstlane(which.y);
        const StripPair *at = a.pairs + pair;
        const StripPair p = *at;
        bool swept;
        Ending ending;
        switch (p.c) {
            case 2: swept = sweep_strip<2, P, RECORD, SH, FREE>(a, p, pair, strip, ring, ending); break;
            case 4: swept = sweep_strip<4, P, RECORD, SH, FREE>(a, p, pair, strip, ring, ending); break;
            default: swept = sweep_strip<8, P, RECORD, SH, FREE>(a, p, pair, strip, ring, ending); break;
        }
        if (!swept) {
            if (threadIdx.x == 0 && a.expired) atomicAdd(a.expired, 1);
            return;
        }
        if (ending.mine) finish_pair<FREE>(a, p, at, ending);
    }
}

// The walk, by a whole wave: every lane makes the walk's moves alike, while the lanes load the decisions of the next 64
// cells along the line the walk is on (the diagonal in the aligned layer, up the column in a deletion layer, along the
// row in an insertion layer), so a round costs one load's latency for up to 64 moves. A move off that line ends the
// round. Lane 0 keeps the moves. One piece by the group sweep's nibbles (walk_tiles' rule), two by the wave sweep's
// flag bytes (walk_rows2's).
template <int P>
__global__ __launch_bounds__(64) void strip_walk(StripArgs a) {
    const int lane = threadIdx.x;
    const SweepArgs &s = a.s;
    const StripPair *at = a.pairs + blockIdx.x;
    const StripPair p = *at;
    const int slot = p.slot;
    int64_t moves = -1;
    if (s.status[slot] == 0 && s.walk_class[slot] == CLASS_STRIP_FIRST &&
        s.walk_flags[slot] == reinterpret_cast<uint64_t>(at) && s.cost[slot] <= s.cap) {
        const int n = s.free_ends ? s.view_rows[slot] : s.tape.rows[slot];
        OpTape ops = op_tape(s, slot);
        const uint32_t unequal = s.eqx ? 1u : 0u;
        int r = s.free_ends ? s.end_row[slot] : n;
        int c = s.free_ends ? s.end_col[slot] : s.tape.cols[slot];
        int layer = 0;
        const int width = strip_columns(p.c);
        while (r > 0 && c > 0) {
            const int dr = (layer == 0 || (layer & 1)) ? 1 : 0;
            const int dc = (layer == 0 || !(layer & 1)) ? 1 : 0;
            const int lr = r - lane * dr, lc = c - lane * dc;
            uint32_t flag = 0;
            if (lr > 0 && lc > 0) {
                const int strip = (lc - 1) / width, within = (lc - 1) % width;
                const int row = lr - strip_first_row(p, strip);
                if (row >= 0 && row < p.rows) {  // a proven band holds the walk; past it the lanes only look ahead
                    const size_t line = ((size_t)strip * p.rows + row) * 64 + within / p.c;
                    const int cell = within % p.c;
                    const uint8_t *record = a.decisions + p.decision_at + line * strip_record_bytes(p.c, P);
                    if (P == 1) flag = (record[cell >> 1] >> (4 * (cell & 1))) & 15u;
                    else flag = record[cell];
                }
            }
            for (int step = 0; step < 64 && r > 0 && c > 0; ++step) {
                const uint32_t f = __builtin_amdgcn_readlane(flag, step);
                uint32_t code;
                if (P == 1) {
                    if ((layer == 1 && (f & 2u)) || (layer == 2 && (f & 1u))) layer = 0;  // the gap opened here
                    if (layer == 0) {
                        const uint32_t stored = f >> 2;  // 3 two unequal letters, 0 deletion, 1 insertion, 2 two equal
                        code = stored == 2 ? 0u : (stored == 3 ? unequal : stored + 2);
                        layer = stored < 2 ? (int)stored + 1 : 0;
                    } else {
                        code = (uint32_t)layer + 1;
                    }
                } else {
                    bool aligned = false;
                    code = 0;
                    if (layer == 0) {
                        const uint32_t src = f & 7u;
                        aligned = src == 0 || src == 5;
                        if (aligned) code = src == 0 ? 0u : unequal;
                        else layer = (int)src;
                    }
                    if (!aligned) {
                        code = (layer & 1) ? 2u : 3u;
                        if (!((f >> (layer + 2)) & 1u)) layer = 0;
                    }
                }
                const int mr = code != 3u, mc = code != 2u;
                if (lane == 0) ops.put(code);
                r -= mr;
                c -= mc;
                if (mr != dr || mc != dc) break;  // off the loaded line
            }
        }
        if (lane == 0) {
            for (; r > 0; --r) ops.put(2u);
            for (; c > 0; --c) ops.put(3u);
            ops.close();
            moves = ops.count;
        }
    }
    publish_cigars(s, slot, moves);
}

__global__ __launch_bounds__(256) void collect_unsettled(const int32_t *status, int slots, int32_t *list,
                                                         int32_t *count) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < slots && status[t] != 0) list[atomicAdd(count, 1)] = t;
}

template <int P, bool SH, bool FREE>
void launch_as(const StripArgs &a, hipStream_t stream) {
    const dim3 grid(a.strips < STRIP_GRID ? a.strips : STRIP_GRID), block(64);
    if (a.decisions) hipLaunchKernelGGL((strip_sweep<P, true, SH, FREE>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((strip_sweep<P, false, SH, FREE>), grid, block, 0, stream, a);
}

}  // namespace

void launch_strip_sweep(const StripArgs &a, hipStream_t stream) {
    if (a.strips <= 0) return;
    const bool shifted = a.s.costs.pieces != 2 && a.s.costs.del_ext == a.s.costs.ins_ext;
    if (a.s.costs.pieces == 2) {
        if (a.s.free_ends) launch_as<2, false, true>(a, stream);
        else launch_as<2, false, false>(a, stream);
    } else if (shifted) {
        if (a.s.free_ends) launch_as<1, true, true>(a, stream);
        else launch_as<1, true, false>(a, stream);
    } else {
        if (a.s.free_ends) launch_as<1, false, true>(a, stream);
        else launch_as<1, false, false>(a, stream);
    }
}

void launch_strip_walk(const StripArgs &a, hipStream_t stream) {
    if (a.count <= 0) return;
    if (a.s.costs.pieces == 2)
        hipLaunchKernelGGL(strip_walk<2>, dim3(a.count), dim3(64), 0, stream, a);
    else
        hipLaunchKernelGGL(strip_walk<1>, dim3(a.count), dim3(64), 0, stream, a);
}

void launch_collect_unsettled(const int32_t *status, int slots, int32_t *list, int32_t *count, hipStream_t stream) {
    if (slots <= 0) return;
    hipLaunchKernelGGL(collect_unsettled, dim3((slots + 255) / 256), dim3(256), 0, stream, status, slots, list, count);
}

}  // namespace dinara
