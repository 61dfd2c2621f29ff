"""The strip sweep (strip.hip) where a pair takes several strips and lanes hold two, four or eight columns: free ends,
whose best end is the least over the strips, and banded rounds keeping decisions, against the oracle bit for bit (cost,
CIGAR and spans; reference tests/test_alignment.mojo:1944-2113 for the free ends' rule, :3715-3989 for the pairs). A
strip is 64 lanes of 2, 4 or 8 columns: queries lie on both sides of 128, 256 and 512 letters and run to several strips.
"""

import ctypes
import random

import pytest

import dinara_align as da
from dinara_align import _lib
from dinara_align.types import UNBOUNDED
from oracle import oracle as o
from test_gpu_costs import mutated
from test_gpu_whole import to_oracle

pytestmark = pytest.mark.gpu

TWO = da.Costs.two_piece(4, 6, 2, 24, 1)
COSTS = [da.Costs.affine(4, 6, 2), TWO, da.Costs.affine(4, 2, 1).with_deletions(6, 3)]
IDS = ["affine", "two-piece", "deletions"]
QUERIES = (127, 128, 129, 255, 256, 257, 511, 513, 769, 1500)


def letters(rng, count, alphabet="ACGT"):
    return "".join(rng.choice(alphabet) for _ in range(count))


def ends_of(mode):
    return (mode.reference_start, mode.reference_end, mode.query_start, mode.query_end)


def free_pairs(rng):
    """(reference, query, mode) with the best end in the last strip, in an earlier one (free query ends), and equal ends
    in different strips (repeats)."""
    found = []
    for m in QUERIES:
        q = letters(rng, m)
        placed = letters(rng, rng.randint(0, 150)) + mutated(q, 0.05, rng) + letters(rng, rng.randint(0, 150))
        if len(placed) + m < 2040:  # the first band, every diagonal a path may start or end on, is 2,048 at most
            found.append((placed, q, da.Mode.INFIX))
        found.append((mutated(q, 0.03, rng) + letters(rng, 90), q, da.Mode.PREFIX))
        found.append((letters(rng, 90) + mutated(q, 0.03, rng), q, da.Mode.SUFFIX))
        # The query's first letters, its middle and its last: ends along the last row, in any strip.
        for low in (0, m // 3, m - m // 4):
            part = mutated(q[low:low + max(20, m // 4)], 0.04, rng)
            found.append((part, q, da.Mode.ends_free(0, 0, UNBOUNDED, UNBOUNDED)))
            found.append((part, q, da.Mode.ends_free(7, 5, UNBOUNDED, UNBOUNDED)))
        # A repeat as long as the query: as many equal ends as copies.
        unit = letters(rng, rng.randint(3, 40))
        found.append(((unit * 8)[:90], (unit * m)[:m], da.Mode.ends_free(0, 0, UNBOUNDED, UNBOUNDED)))
        found.append(((unit * m)[:m + 100], (unit * m)[:m], da.Mode.ends_free(50, 50, 20, 20)))
    return found


@pytest.mark.parametrize("columns", [None, "2", "8"])
@pytest.mark.parametrize("costs", COSTS, ids=IDS)
def test_free_ends_across_strips(costs, columns, monkeypatch):
    if columns:
        monkeypatch.setenv("DINARA_STRIP_COLUMNS", columns)
    rng = random.Random(101 + len(str(costs)))
    oc = to_oracle(costs)
    by_mode = {}
    for r, q, mode in free_pairs(rng):
        by_mode.setdefault(ends_of(mode), (mode, [], []))
        by_mode[ends_of(mode)][1].append(r)
        by_mode[ends_of(mode)][2].append(q)
    for ends, (mode, refs, qrys) in by_mode.items():
        for ties in ("left", "right"):
            got = da.alignments(refs, qrys, costs, mode, ties=ties)
            for i, (r, q) in enumerate(zip(refs, qrys)):
                g = got[i]
                assert g is not None, (i, len(r), len(q), mode, ties)
                assert (g.cost, g.cigar, (g.reference_start, g.reference_end, g.query_start, g.query_end)) == o.ends_align(
                    r, q, oc, ends, right_ties=ties == "right"), (i, len(r), len(q), mode, ties)
        assert da.distances(refs, qrys, costs, mode) == [o.ends_cost(r, q, oc, ends)[0] for r, q in zip(refs, qrys)]


@pytest.mark.parametrize("columns", ["2", "4", "8"])
@pytest.mark.parametrize("costs", COSTS, ids=IDS)
def test_banded_strips_of_every_width(costs, columns, monkeypatch):
    # Bands far narrower than the matrix: strips whose rows begin below the first and end above the last, the cell
    # above-left of a strip's first from the strip to its left, and decisions in the rows between.
    monkeypatch.setenv("DINARA_STRIP_COLUMNS", columns)
    rng = random.Random(7)
    oc = to_oracle(costs)
    refs, qrys = [], []
    for n, rate in [(4100, 0.002), (4100, 0.03), (2300, 0.05), (3000, 0.25), (2600, 0.6), (1300, 0.1)]:
        r = letters(rng, n)
        refs.append(r)
        qrys.append(mutated(r, rate, rng))
    refs += [letters(rng, 3000), letters(rng, 900), "ACG" * 1000]
    qrys += [refs[-3][400:2500], letters(rng, 300) + refs[-2] + letters(rng, 1400), "ACG" * 600 + "TTAC" * 300]
    refs += ["", letters(rng, 700)]
    qrys += [letters(rng, 700), ""]
    for ties in ("left", "right"):
        got = da.alignments(refs, qrys, costs, ties=ties)
        for i, (r, q) in enumerate(zip(refs, qrys)):
            assert (got[i].cost, got[i].cigar) == o.costs_align(r, q, oc, right_ties=ties == "right"), (i, len(r), len(q))
    assert da.distances(refs, qrys, costs) == [o.costs_cost(r, q, oc) for r, q in zip(refs, qrys)]


@pytest.mark.parametrize("free", [None, da.Mode.ends_free(4, 3, 2, 5), da.Mode.PREFIX])
@pytest.mark.parametrize("costs", COSTS[:2], ids=IDS[:2])
def test_narrow_wave_bands_and_wider(costs, free):
    # Under two pieces or free ends short pairs take wave bands of 64 diagonals and 128 (128 under free ends up to 320
    # letters, the narrower up to the pairs' mean at least), others strips: first bands of 62 to 66 and 126 to 130
    # diagonals, retries into each, lengths around the limits.
    rng = random.Random(29)
    refs, qrys = [], []
    for difference in (0, 1, 58, 59, 60, 61, 62, 63, 64, 122, 123, 124, 125, 126, 127, 128):
        for m in (30, 96, 97, 190):
            q = letters(rng, m)
            cut = rng.randint(0, m)
            refs.append(mutated(q[:cut], 0.05, rng) + letters(rng, difference) + q[cut:])
            qrys.append(q)
    for n, rate in [(150, 0.02), (150, 0.3), (255, 0.1), (257, 0.1), (257, 0.5), (400, 0.02), (900, 0.01), (2000, 0.002)]:
        for _ in range(3):
            r = letters(rng, n)
            refs.append(r)
            qrys.append(mutated(r, rate, rng))
    refs += ["", "ACGT", ""]
    qrys += ["ACG", "", ""]
    oc, ends = to_oracle(costs), ends_of(free) if free else (0, 0, 0, 0)
    for ties in ("left", "right"):
        got = da.alignments(refs, qrys, costs, *([free] if free else []), ties=ties)
        for i, (r, q) in enumerate(zip(refs, qrys)):
            g = got[i]
            assert (g.cost, g.cigar, (g.reference_start, g.reference_end, g.query_start, g.query_end)) == o.ends_align(
                r, q, oc, ends, right_ties=ties == "right"), (i, len(r), len(q), ties)
    assert da.distances(refs, qrys, costs, *([free] if free else [])) == [
        o.ends_cost(r, q, oc, ends)[0] for r, q in zip(refs, qrys)]


def resident(refs, qrys, costs, kind, mode=None):
    """A resident batch's results of two runs through the C ABI, the launches of a run and its pairs swept whole."""
    handle = _lib.lib()
    R, Q = _lib.Texts(refs), _lib.Texts(qrys)
    c, status = costs.as_c(), ctypes.c_int64(0)
    as_c = mode.as_c() if mode else None
    batch = handle.dinara_batch_new(0, kind, len(refs), *R.args(), *Q.args(), ctypes.byref(c),
                                    ctypes.byref(as_c) if mode else None, None, 4, ctypes.byref(status))
    assert batch, status.value
    try:
        runs = []
        for _ in range(2):
            assert handle.dinara_batch_run(batch) == 0
            if kind == _lib.BATCH_DISTANCES:
                out = (ctypes.c_int64 * len(refs))()
                assert handle.dinara_batch_distances(batch, out) == 0
                runs.append(list(out))
                continue
            found, statuses = (_lib.CAlignment * len(refs))(), (ctypes.c_int64 * len(refs))()
            assert handle.dinara_batch_alignments(batch, found, statuses) == 0
            assert not any(statuses)
            runs.append([(a.cost, ctypes.string_at(a.cigar, a.cigar_length).decode()) for a in found])
            for a in found:
                handle.dinara_free(a.cigar)
        assert runs[0] == runs[1]
        return runs[0], handle.dinara_batch_stat(batch, 2), handle.dinara_batch_stat(batch, 10)
    finally:
        handle.dinara_batch_free(batch)


@pytest.mark.parametrize("costs", COSTS, ids=IDS)
def test_rounds_cut_into_parts(costs, monkeypatch):
    # A round whose memory passes its budget runs in parts, each reusing the memory of the one before: costs alone
    # (whose carry records are all they keep), CIGARs, and the two phases of free ends.
    rng = random.Random(19)
    oc = to_oracle(costs)
    refs = [letters(rng, rng.randint(2200, 2700)) for _ in range(24)]
    qrys = [mutated(r, rate, rng) for r, rate in zip(refs, [0.01, 0.1, 0.3, 0.5] * 6)]
    windows = [letters(rng, 60) + q[:600] + letters(rng, 90) for q in qrys]
    reads = [mutated(q[:600], 0.05, rng) for q in qrys]
    want = [o.costs_align(r, q, oc) for r, q in zip(refs, qrys)]
    ends = [o.ends_align(r, q, oc, ends_of(da.Mode.INFIX)) for r, q in zip(windows, reads)]
    whole = {}
    for budget in (None, 300_000, 1):
        if budget:
            monkeypatch.setenv("DINARA_STRIP_BUDGET", str(budget))
        for name, got, right in [
                ("distances", resident(refs, qrys, costs, 0), [cost for cost, _ in want]),
                ("alignments", resident(refs, qrys, costs, 1), want),
                ("placed distances", resident(windows, reads, costs, 0, da.Mode.INFIX), [e[0] for e in ends]),
                ("placed", resident(windows, reads, costs, 1, da.Mode.INFIX), [e[:2] for e in ends])]:
            assert got[0] == right, (name, budget)
            launches = whole.setdefault(name, got[1])
            assert budget is None or got[1] > launches, (name, budget, got[1], launches)


@pytest.mark.parametrize("costs", COSTS, ids=IDS)
def test_pairs_of_expired_waits_are_swept_whole(costs, monkeypatch):
    # Waits that give up at once (as one would after seconds): every kernel ends, and the pairs that leaves unsettled,
    # all of them short enough for a band to settle, take the whole-matrix path.
    rng = random.Random(23)
    oc = to_oracle(costs)
    refs = [letters(rng, rng.randint(2200, 2700)) for _ in range(12)] + [letters(rng, 90) for _ in range(20)]
    qrys = [mutated(r, rate, rng) for r, rate in zip(refs, [0.01, 0.1, 0.3, 0.5] * 8)]
    want = [o.costs_align(r, q, oc) for r, q in zip(refs, qrys)]
    assert resident(refs, qrys, costs, 1)[2] == 0
    monkeypatch.setenv("DINARA_STRIP_POLLS", "0")
    for kind in (0, 1):
        got, _, whole = resident(refs, qrys, costs, kind)
        assert got == (want if kind else [cost for cost, _ in want])
        assert whole > 0


def test_first_rounds_after_seeds_and_whole_runs():
    # The first round's strips are planned once while the first bands stand: seeds move them, and a run of whole matrices
    # between two banded ones uses the same memory.
    rng = random.Random(31)
    costs = COSTS[0]
    refs = [letters(rng, rng.randint(2200, 2700)) for _ in range(10)] + [letters(rng, 3000)]
    qrys = [mutated(r, rate, rng) for r, rate in zip(refs, [0.01, 0.1, 0.3, 0.5, 0.02] * 2)] + [refs[-1][900:2100]]
    want = [o.costs_align(r, q, to_oracle(costs)) for r, q in zip(refs, qrys)]
    handle = _lib.lib()
    R, Q, c, status = _lib.Texts(refs), _lib.Texts(qrys), costs.as_c(), ctypes.c_int64(0)
    for kind in (0, 1):
        batch = handle.dinara_batch_new(0, kind, len(refs), *R.args(), *Q.args(), ctypes.byref(c), None, None, 4,
                                        ctypes.byref(status))
        assert batch, status.value
        try:
            for guesses, whole in [(None, 0), (None, 1), (0, 0), (None, 0), (700, 0), (4000, 0), (None, 1), (60, 0)]:
                if guesses is not None:
                    seeds = (ctypes.c_int64 * len(refs))(*[guesses] * len(refs))
                    assert handle.dinara_batch_seed(batch, ctypes.addressof(seeds)) == 0
                assert handle.dinara_batch_set_whole(batch, whole) == 0
                assert handle.dinara_batch_run(batch) == 0
                if kind == 0:
                    out = (ctypes.c_int64 * len(refs))()
                    assert handle.dinara_batch_distances(batch, out) == 0
                    assert list(out) == [cost for cost, _ in want], (guesses, whole)
                    continue
                found, statuses = (_lib.CAlignment * len(refs))(), (ctypes.c_int64 * len(refs))()
                assert handle.dinara_batch_alignments(batch, found, statuses) == 0
                got = [(a.cost, ctypes.string_at(a.cigar, a.cigar_length).decode()) for a in found]
                for a in found:
                    handle.dinara_free(a.cigar)
                assert got == want, (guesses, whole)
        finally:
            handle.dinara_batch_free(batch)


@pytest.mark.parametrize("pairs,length", [(270_000, 100), (60_000, 300)])
def test_plans_larger_than_the_memory_kept_for_them(pairs, length, monkeypatch):
    # Rounds of more than 262,144 pairs, and of more strips (two columns a lane), in one call after another.
    monkeypatch.setenv("DINARA_STRIP_COLUMNS", "2")
    rng = random.Random(length)
    oc = to_oracle(COSTS[0])
    windows = [letters(rng, length + rng.randint(0, 5)) for _ in range(40)]
    reads = [mutated(w, 0.05, rng)[2:] + (letters(rng, 600) if length > 100 and i % 2 else "") for i, w in enumerate(windows)]
    want = [o.ends_align(r, q, oc, ends_of(da.Mode.INFIX)) for r, q in zip(windows, reads)]
    print(f"[strips] {pairs} pairs", flush=True)
    refs, qrys = (windows * (pairs // 40 + 1))[:pairs], (reads * (pairs // 40 + 1))[:pairs]
    assert da.distances(refs, qrys, COSTS[0], da.Mode.INFIX) == ([e[0] for e in want] * (pairs // 40 + 1))[:pairs]
    found = da.alignments(refs[:1000], qrys[:1000], COSTS[0], da.Mode.INFIX)
    assert [(a.cost, a.cigar) for a in found] == ([e[:2] for e in want] * 25)[:1000]
