"""The work this framework is used for, as cases that can be timed: which inputs a caller has, and one pass over them
through the public entry points (the Python package, the C ABI's drop-in calls, its resident batches and its network).

`listed()` names the cases, `draw(rng)` gives further ones of the same ranges, `prepare(case, seed)` makes what a
caller holds before the call, `run(state)` is one pass and returns its results whole, `work(case)` the bytes and
operations a pass cannot do without, and `exact(case, seed)` the network's numbers in 64 bits. Alignment results are
whole numbers and text, which have one right value each.

A case's fields: `path` (costs, scoring or network), `form` (package: the Python calls; call: the C ABI's drop-in call
on letters in host memory; resident: a batch kept on the device, run again and its results copied out), `op`, the
batch (`pairs`, reference letters log-normal around `length` with `sigma`, at most `longest`, at least a tenth of
`length`, mutated at a rate uniform in `low`..`high`), and the options.
"""

import collections
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "dinara-align_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import dinara_align as da  # noqa: E402
from dinara_align import _lib  # noqa: E402
from dinara_align.synthetic import protein_table  # noqa: E402

THREADS = 16        # the packing threads a caller asks for
STRIDE = 288        # floats a feature row
HIDDEN = 256
ALPHABETS = {"dna": b"ACGT", "dna_n": b"ACGTN", "protein": b"ACDEFGHIKLMNPQRSTVWY"}
COSTS = {
    "unit": da.Costs.edit(),
    "affine": da.Costs.affine(4, 6, 2),
    "affine_121": da.Costs.affine(1, 2, 1),
    "affine_51101": da.Costs.affine(5, 11, 1),
    "linear": da.Costs.linear(3, 2),
    "two_piece": da.Costs.two_piece(4, 6, 2, 24, 1),
    "deletions": da.Costs.affine(4, 2, 1).with_deletions(9, 1),
}
MODES = {"global": da.Mode.GLOBAL, "infix": da.Mode.INFIX, "local": da.Mode.local()}
ALIGNMENT = np.dtype([(name, np.int64) for name in ("cost", "score", "reference_start", "reference_end",
                                                    "query_start", "query_end", "cigar", "cigar_length")])
PLAIN = {"sigma": 0.0, "low": 0.02, "high": 0.02, "window": 0, "letters": "dna", "costs": "unit", "mode": "global",
         "ties": "left", "eqx": True, "band": 0, "cap": -1, "learned": False}


def _case(name, path, form, op, pairs, length, **options):
    case = {"name": name, "path": path, "form": form, "op": op, "pairs": pairs, "length": length, **PLAIN, **options}
    case.setdefault("longest", 8 * length)
    return case


def listed():
    return [
        # One read against one section through the Python package: the smallest call, all latency.
        _case("one_read", "costs", "package", "alignments", 1, 150),
        # Edit distances of 10,000 short reads, 150 bp at 2%: the first benchmark configuration's batch.
        _case("reads_edit", "costs", "resident", "distances", 10_000, 150),
        # Unit-cost CIGARs of reads of very different lengths, a caller's first and only call on them.
        _case("uneven_call", "costs", "call", "alignments", 4_000, 1_500, sigma=1.0, longest=20_000, low=0.01,
              high=0.15),
        # The same kind of batch resident, its first bands seeded by the trained network: the headline configuration.
        _case("uneven_learned", "costs", "resident", "alignments", 20_000, 1_500, sigma=1.0, longest=20_000,
              low=0.01, high=0.15, learned=True),
        # Gap-affine distances of Illumina-length reads at 1%: the reference's own published batch workload.
        _case("reads_affine", "costs", "resident", "distances", 200_000, 148, low=0.01, high=0.01, costs="affine"),
        # Gap-affine CIGARs of 250 bp reads at 5% in one drop-in call: the second configuration's pairs.
        _case("reads_affine_call", "costs", "call", "alignments", 20_000, 250, low=0.05, high=0.05, costs="affine"),
        # Gap-affine distances of long and short reads mixed: the fourth configuration's pairs.
        _case("uneven_affine", "costs", "resident", "distances", 2_000, 1_500, sigma=1.0, longest=20_000, low=0.01,
              high=0.15, costs="affine"),
        # Two-piece gap costs over noisy long-read pieces, CIGARs.
        _case("two_piece", "costs", "resident", "alignments", 1_000, 1_500, sigma=0.4, longest=5_000, low=0.03,
              high=0.10, costs="two_piece"),
        # Reads placed inside a wider window (free reference ends), gap-affine, CIGARs and spans.
        _case("infix_reads", "costs", "resident", "alignments", 5_000, 200, sigma=0.2, longest=400, low=0.02,
              high=0.06, window=600, costs="affine", mode="infix"),
        # Global scores of short reads under a substitution table, the published batch workload's device form.
        _case("reads_scores", "scoring", "resident", "scores", 100_000, 148, low=0.01, high=0.01, costs="dna"),
        # Local protein alignments, 300 residues against windows of 3,000: the fifth configuration's pairs.
        _case("local_protein", "scoring", "resident", "alignments", 5_000, 300, low=0.30, high=0.30, window=3_000,
              letters="protein", costs="protein", mode="local"),
        # Training the band network as a caller does before seeding with it: shuffled batches, Adam.
        {"name": "train", "path": "network", "op": "train", "rows": 32_768, "length": 1_000, "batch": 4_096,
         "epochs": 2},
    ]


def draw(rng):
    def size(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    def rate(low, high):
        return round(rng.uniform(low, high), 4)

    kind = rng.randrange(12)
    if kind == 0:
        return _drawn("costs", "package", rng.choice(["distances", "alignments"]), size(1, 64), size(20, 400), rng,
                      low=rate(0.0, 0.05), high=0.1, costs=rng.choice(["unit", "affine", "linear"]))
    if kind == 1:
        return _drawn("costs", rng.choice(["resident", "call"]), "distances", size(500, 10_000), size(50, 151), rng,
                      sigma=rate(0.0, 0.3), high=rate(0.02, 0.1), letters=rng.choice(["dna", "dna", "dna_n"]),
                      cap=rng.choice([-1, -1, 8]))
    if kind == 2:
        return _drawn("costs", "call", "alignments", size(100, 3_000), size(200, 1_500), rng, sigma=rate(0.2, 0.9),
                      longest=12_000, low=0.01, high=rate(0.05, 0.15))
    if kind == 3:
        return _drawn("costs", "resident", "alignments", size(1_000, 15_000), size(400, 1_500), rng,
                      sigma=rate(0.3, 0.9), longest=15_000, low=0.01, high=rate(0.05, 0.15), learned=True)
    if kind == 4:
        return _drawn("costs", "resident", "distances", size(5_000, 200_000), size(75, 148), rng,
                      sigma=rate(0.0, 0.1), low=0.005, high=rate(0.01, 0.03),
                      costs=rng.choice(["affine", "affine_121", "linear"]))
    if kind == 5:
        return _drawn("costs", rng.choice(["call", "resident"]), "alignments", size(500, 20_000), size(100, 250), rng,
                      sigma=rate(0.0, 0.1), low=0.01, high=rate(0.03, 0.08), eqx=rng.random() < 0.7,
                      costs=rng.choice(["affine", "affine", "deletions", "affine_51101"]),
                      band=rng.choice([0, 0, 0, 40]))
    if kind == 6:
        return _drawn("costs", "resident", rng.choice(["distances", "alignments"]), size(50, 1_000),
                      size(500, 1_500), rng, sigma=rate(0.2, 0.7), longest=8_000, low=0.01, high=rate(0.05, 0.12),
                      costs="affine")
    if kind == 7:
        return _drawn("costs", "resident", rng.choice(["distances", "alignments"]), size(50, 1_000),
                      size(150, 1_500), rng, sigma=rate(0.0, 0.4), longest=4_000, low=0.02, high=rate(0.03, 0.10),
                      costs="two_piece")
    if kind == 8:
        return _drawn("costs", "resident", rng.choice(["distances", "alignments"]), size(200, 5_000), size(60, 200),
                      rng, sigma=rate(0.0, 0.2), longest=400, low=0.01, high=rate(0.02, 0.06), window=size(200, 600),
                      costs=rng.choice(["affine", "affine", "unit", "two_piece"]), mode="infix")
    if kind == 9:
        return _drawn("scoring", "resident", rng.choice(["scores", "scores", "alignments"]), size(1_000, 50_000),
                      size(50, 250), rng, sigma=rate(0.0, 0.2), low=0.01, high=rate(0.02, 0.1),
                      costs=rng.choice(["dna", "dna_default", "protein"]))
    if kind == 10:
        return _drawn("scoring", rng.choice(["resident", "call"]), rng.choice(["scores", "alignments"]),
                      size(200, 5_000), size(80, 300), rng, sigma=rate(0.0, 0.3), longest=600, low=0.1, high=0.35,
                      window=size(400, 2_500), letters="protein", costs="protein", mode="local")
    case = {"path": "network", "op": rng.choice(["train", "gradients", "predict"]), "rows": size(1_000, 32_768),
            "length": size(300, 1_000), "batch": 32 * size(8, 128), "epochs": rng.randint(1, 2)}
    return case


def _drawn(path, form, op, pairs, length, rng, **options):
    case = _case("", path, form, op, pairs, length, **options)
    del case["name"]
    case["high"] = max(case["low"], case["high"])
    if path == "scoring":
        case["letters"] = "protein" if case["costs"] == "protein" else "dna"
    elif op == "alignments" and case["mode"] == "global":
        case["ties"] = rng.choice(["left", "left", "right"])
    return case


# ------------------------------------------------------------------ inputs

def _generator(seed, device):
    return torch.Generator(device=device).manual_seed(int(seed) * 7919 + 17)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _starts(lengths):
    return torch.cumsum(lengths, 0) - lengths


def _pairs(case, seed):
    """The batch's sequences as letter codes on the device: (reference codes, lengths, query codes, lengths, events a
    pair). A letter is substituted, has letters inserted before it or is deleted; runs of indels are geometric (0.7)
    under gap costs, one letter under unit costs."""
    device = _device()
    g = _generator(seed, device)
    pairs, length, alphabet = case["pairs"], case["length"], len(ALPHABETS[case["letters"]])

    def uniform(*shape):
        return torch.rand(*shape, generator=g, device=device)

    def letters(count):
        return torch.randint(0, alphabet, (int(count),), generator=g, device=device, dtype=torch.uint8)

    spread = torch.randn(pairs, generator=g, device=device) * case["sigma"]
    lengths = torch.clamp(torch.round(length * torch.exp(spread)), max(1, length // 10), case["longest"]).long()
    rates = case["low"] + uniform(pairs) * (case["high"] - case["low"])
    owner = torch.repeat_interleave(torch.arange(pairs, device=device), lengths)
    codes = letters(len(owner))
    if case["letters"] == "dna_n":  # an N here and there
        codes = torch.where(uniform(len(codes)) < 0.998, codes % 4, torch.full_like(codes, 4))
    event = uniform(len(codes)) < rates[owner]
    kind = uniform(len(codes))
    swap, insert, delete = event & (kind < 0.6), event & (kind >= 0.6) & (kind < 0.8), event & (kind >= 0.8)
    run = torch.ones_like(owner)
    if case["costs"] != "unit":
        run = 1 + torch.floor(torch.log(uniform(len(codes)).clamp_min(1e-7)) / math.log(0.3)).long()
    # Deleted runs end at their pair's end.
    place = torch.arange(len(codes), device=device)
    end = (torch.cumsum(lengths, 0))[owner]
    cover = torch.zeros(len(codes) + 1, dtype=torch.int32, device=device)
    at = place[delete]
    cover.index_add_(0, at, torch.ones_like(at, dtype=torch.int32))
    cover.index_add_(0, torch.minimum(at + run[delete], end[delete]), -torch.ones_like(at, dtype=torch.int32))
    gone = torch.cumsum(cover[:-1], 0) > 0
    mutated = torch.where(swap, (codes + 1 + letters(len(codes)) % (alphabet - 1)) % alphabet, codes)
    copies = torch.where(gone, 0, 1) + torch.where(insert & ~gone, run, 0)
    source = torch.repeat_interleave(place, copies)
    last = torch.cumsum(copies, 0)[source] - 1  # a letter's own copy comes last, the inserted ones before it
    fresh = torch.arange(len(source), device=device) != last
    query = torch.where(fresh, letters(len(source)), mutated[source])
    query_lengths = torch.zeros(pairs, dtype=torch.int64, device=device).index_add_(0, owner, copies)
    events = torch.zeros(pairs, dtype=torch.int64, device=device).index_add_(0, owner, event.long())
    if case["window"]:
        # The mutated copy at a random place of a random window, against the unmutated sequence.
        window = case["window"]
        wide = torch.maximum(query_lengths, torch.full_like(query_lengths, window))
        offset = torch.floor(uniform(pairs) * (wide - query_lengths + 1)).long()
        text = letters(wide.sum())
        query_owner = torch.repeat_interleave(torch.arange(pairs, device=device), query_lengths)
        within = torch.arange(len(query), device=device) - _starts(query_lengths)[query_owner]
        text[_starts(wide)[query_owner] + offset[query_owner] + within] = query
        return text, wide, codes, lengths, events
    return codes, lengths, query, query_lengths, events


class _Texts:
    """A batch's sequences in host memory as the C ABI takes them: first bytes and lengths."""

    def __init__(self, codes, lengths, alphabet):
        table = torch.tensor(list(alphabet), dtype=torch.uint8, device=codes.device)
        self.letters = np.ascontiguousarray(table[codes.long()].cpu().numpy())
        self.lengths = np.ascontiguousarray(lengths.cpu().numpy().astype(np.int64))
        first = np.cumsum(self.lengths) - self.lengths
        self.pointers = np.ascontiguousarray(first.astype(np.uint64) + np.uint64(self.letters.ctypes.data))
        self.first = first

    def args(self):
        return self.pointers.ctypes.data, self.lengths.ctypes.data

    def as_bytes(self):
        text = self.letters.tobytes()
        return [text[a:a + n] for a, n in zip(self.first.tolist(), self.lengths.tolist())]


class _Held:
    """A handle of the library's, given back when the state holding it goes."""

    def __init__(self, value, give_back):
        self.value, self.give_back = value, give_back

    def __del__(self):
        if self.value:
            self.give_back(self.value)
            self.value = None


def _scoring(case):
    if case["costs"] == "protein":
        alphabet, table = protein_table()
        return da.Scoring.tabulated(alphabet, table, -11, -1)
    if case["costs"] == "dna_default":
        return da.Scoring.dna()
    return da.Scoring.uniform(0, -1, -2, -1)


def _check(code):
    if code != 0:
        raise RuntimeError("the library returned code %d" % code)


def prepare(case, seed):
    if case["path"] == "network":
        return _prepare_network(case, seed)
    codes, lengths, query, query_lengths, _ = _pairs(case, seed)
    alphabet = ALPHABETS[case["letters"]]
    refs, qrys = _Texts(codes, lengths, alphabet), _Texts(query, query_lengths, alphabet)
    state = {"case": case, "handle": _lib.lib()}
    if case["op"] == "alignments":
        state["text"] = np.zeros(_text_room(case), np.uint8)
    if case["form"] == "package":
        state["refs"], state["qrys"] = refs.as_bytes(), qrys.as_bytes()
        return state
    pairs = case["pairs"]
    state.update(refs=refs, qrys=qrys, numbers=np.zeros(pairs, np.int64), statuses=np.zeros(pairs, np.int64),
                 found=np.zeros(pairs, ALIGNMENT), mode=MODES[case["mode"]].as_c())
    if case["path"] == "scoring":
        state["scoring"], state["kept"] = _scoring(case).as_c()
    else:
        state["costs"] = COSTS[case["costs"]].as_c()
        band = case["band"]
        state["options"] = _lib.COptions(band_low=-band if band else -(1 << 63), band_high=band if band else (1 << 63) - 1,
                                         max_cost=case["cap"], eqx=int(case["eqx"]),
                                         right_ties=int(case["ties"] == "right"), max_memory=0)
    if case["form"] == "resident":
        state["batch"] = _resident(case, state)
    return state


def _resident(case, state):
    handle, status = state["handle"], ctypes.c_int64(0)
    kind = _lib.BATCH_ALIGNMENTS if case["op"] == "alignments" else _lib.BATCH_DISTANCES
    head = (0, kind, case["pairs"], *state["refs"].args(), *state["qrys"].args())
    if case["path"] == "scoring":
        batch = handle.dinara_scoring_batch_new(*head, ctypes.byref(state["scoring"]), ctypes.byref(state["mode"]),
                                                int(case["eqx"]), THREADS, ctypes.byref(status))
        free = handle.dinara_scoring_batch_free
    else:
        batch = handle.dinara_batch_new(*head, ctypes.byref(state["costs"]), ctypes.byref(state["mode"]),
                                        ctypes.byref(state["options"]), THREADS, ctypes.byref(status))
        free = handle.dinara_batch_free
    if not batch:
        raise RuntimeError("no batch: code %d" % status.value)
    if case["learned"]:
        state["net"] = _trained()
        _check(handle.dinara_batch_set_keep_first(batch, 1))
        _check(handle.dinara_batch_set_graph(batch, 0))
    return _Held(batch, free)


_NET = []


def _trained():
    """A program trains its network once and seeds every batch with it: 24,000 pairs, their labels the aligner's own
    costs."""
    if not _NET:
        handle = _lib.lib()
        case = _case("", "costs", "resident", "distances", 24_000, 1_500, sigma=0.9, longest=20_000, low=0.01,
                     high=0.15)
        state = prepare(case, 424242)
        costs, batch = run(state), state["batch"].value
        rows = np.zeros((case["pairs"], STRIDE), np.float32)
        _check(handle.dinara_batch_features(batch, rows.ctypes.data))
        targets = np.log1p(np.maximum(costs, 0)).astype(np.float32)
        net = _Held(handle.dinara_mlp_new(0, 17), handle.dinara_mlp_free)
        _check(handle.dinara_mlp_train(net.value, len(rows), rows.ctypes.data, targets.ctypes.data, 6, 512, 2e-3, 7,
                                       None))
        _NET.append(net)
    return _NET[0]


def _weights(seed):
    """A network's weights as training starts from them, flat: w1, b1, w2, b2, w3, b3."""
    g = torch.Generator().manual_seed(int(seed) * 104729 + 5)
    w1 = torch.randn(STRIDE, HIDDEN, generator=g) * math.sqrt(2 / 258)
    w1[258:] = 0
    w2 = torch.randn(HIDDEN, HIDDEN, generator=g) * math.sqrt(2 / HIDDEN)
    w3 = torch.randn(HIDDEN, generator=g) * math.sqrt(1 / HIDDEN)
    zeros = torch.zeros(HIDDEN)
    return torch.cat([w1.reshape(-1), zeros, w2.reshape(-1), zeros, w3, torch.tensor([7.0])]).float()


def _rows(case, seed):
    """Feature rows and targets of pairs like those a caller trains on: 4-mer count differences and lengths, and the
    logarithm of the pair's edits."""
    pairs = _case("", "costs", "resident", "distances", case["rows"], case["length"], sigma=0.8,
                  longest=6 * case["length"], low=0.01, high=0.15)
    codes, lengths, query, query_lengths, events = _pairs(pairs, seed)

    def counts(letters, sizes):
        owner = torch.repeat_interleave(torch.arange(len(sizes), device=letters.device), sizes)
        c = letters.long()
        word = c[:-3] * 64 + c[1:-2] * 16 + c[2:-1] * 4 + c[3:]
        whole = owner[3:] == owner[:-3]
        return torch.bincount(owner[3:][whole] * 256 + word[whole], minlength=256 * len(sizes)).reshape(-1, 256)

    n, m = lengths.float(), query_lengths.float()
    x = torch.zeros(case["rows"], STRIDE, device=codes.device)
    x[:, :256] = (counts(codes, lengths) - counts(query, query_lengths)) * (8 / torch.sqrt(1 + n + m))[:, None]
    x[:, 256] = (torch.log1p(n) - 7) / 2
    x[:, 257] = (torch.log1p(m) - 7) / 2
    return x, torch.log1p(events.float())


def _prepare_network(case, seed):
    x, y = _rows(case, seed)
    state = {"case": case, "handle": _lib.lib(), "x": np.ascontiguousarray(x.cpu().numpy()),
             "y": np.ascontiguousarray(y.cpu().numpy()), "weights": _weights(seed).numpy(),
             "out": np.zeros(case["rows"], np.float32)}
    if case["op"] != "train":
        net = state["handle"].dinara_mlp_new(0, 17)
        state["net"] = _Held(net, state["handle"].dinara_mlp_free)
        _check(state["handle"].dinara_mlp_set_weights(net, state["weights"].ctypes.data))
        state["gradients"] = np.zeros(len(state["weights"]), np.float32)
    return state


# ------------------------------------------------------------------ one pass

def run(state):
    case = state["case"]
    if case["path"] == "network":
        return _run_network(state)
    if case["form"] == "package":
        costs, mode = COSTS[case["costs"]], MODES[case["mode"]]
        if case["op"] == "distances":
            return np.array(da.distances(state["refs"], state["qrys"], costs, mode), np.int64)
        found = da.alignments(state["refs"], state["qrys"], costs, mode, ties=case["ties"], eqx=case["eqx"])
        texts = [a.cigar for a in found]
        _keep(state, "".join(texts).encode())
        return {"cost": np.array([a.cost for a in found], np.int64),
                "length": np.array([len(t) for t in texts], np.int64), "cigar": state["text"]}
    handle, refs, qrys = state["handle"], state["refs"], state["qrys"]
    numbers, found, statuses = state["numbers"].ctypes.data, state["found"].ctypes.data, state["statuses"]
    aligned = case["op"] == "alignments"
    if case["form"] == "call":
        head = (0, case["pairs"], *refs.args(), *qrys.args())
        if case["path"] == "scoring":
            head += (ctypes.byref(state["scoring"]), ctypes.byref(state["mode"]))
            if aligned:
                code = handle.dinara_gpu_scoring_alignments(*head, int(case["eqx"]), THREADS, found, _at(statuses))
            else:
                code = handle.dinara_gpu_scores(*head, THREADS, _at(state["numbers"]))
        else:
            head += (ctypes.byref(state["costs"]), ctypes.byref(state["mode"]), ctypes.byref(state["options"]))
            if aligned:
                code = handle.dinara_gpu_alignments(*head, THREADS, found, _at(statuses))
            else:
                code = handle.dinara_gpu_distances(*head, THREADS, _at(state["numbers"]))
        _check(code)
    else:
        batch = state["batch"].value
        if case["path"] == "scoring":
            _check(handle.dinara_scoring_batch_run(batch))
            if aligned:
                _check(handle.dinara_scoring_batch_alignments(batch, refs.args()[0], qrys.args()[0], found,
                                                              _at(statuses)))
            else:
                _check(handle.dinara_scoring_batch_scores(batch, _at(state["numbers"])))
        else:
            if case["learned"]:
                _check(handle.dinara_batch_seed_learned_by_length(batch, state["net"].value, 0.0, 0.1))
            _check(handle.dinara_batch_run(batch))
            if aligned:
                _check(handle.dinara_batch_alignments(batch, found, _at(statuses)))
            else:
                _check(handle.dinara_batch_distances(batch, _at(state["numbers"])))
    if not aligned:
        return state["numbers"]
    return _read(state)


def _at(array):
    return ctypes.cast(array.ctypes.data, ctypes.POINTER(ctypes.c_int64))


def _read(state):
    """The call's alignments as a program reads them, each CIGAR then freed."""
    found, statuses = state["found"], state["statuses"]
    if statuses.any():  # a refused pair's fields are left as they were
        found[statuses != 0] = 0
    pointers = np.ascontiguousarray(found["cigar"])
    texts = (ctypes.c_char_p * len(pointers)).from_buffer(pointers)[:]
    _keep(state, b"".join(filter(None, texts)))
    collections.deque(map(state["handle"].dinara_free, pointers.tolist()), maxlen=0)
    return {"status": statuses, "cigar": state["text"],
            **{name: found[name].copy() for name in ALIGNMENT.names if name != "cigar"}}


def _text_room(case):
    """Room for a batch's CIGARs one after another: about five letters an edit, and as much again to spare."""
    edits = _letters(case)[1] * (case["low"] + case["high"]) / 2
    return 1 << 16 if case["pairs"] <= 64 else (1 << 18) + int(case["pairs"] * (16 + 10 * edits))


def _keep(state, text):
    """The batch's CIGARs in the program's own buffer, zeros after them."""
    room, before = state["text"], state.get("used", 0)
    room[:len(text)] = np.frombuffer(text, np.uint8)
    room[len(text):before] = 0
    state["used"] = len(text)


def _run_network(state):
    case, handle = state["case"], state["handle"]
    rows, x, y = case["rows"], state["x"].ctypes.data, state["y"].ctypes.data
    loss = ctypes.c_double(0)
    if case["op"] == "train":
        net = _Held(handle.dinara_mlp_new(0, 17), handle.dinara_mlp_free)
        weights = np.empty(len(state["weights"]), np.float32)
        _check(handle.dinara_mlp_set_weights(net.value, state["weights"].ctypes.data))
        _check(handle.dinara_mlp_train(net.value, rows, x, y, case["epochs"], case["batch"], 2e-3, 7,
                                       ctypes.byref(loss)))
        _check(handle.dinara_mlp_get_weights(net.value, weights.ctypes.data))
        return {"weights": weights, "loss": float(loss.value)}
    if case["op"] == "predict":
        _check(handle.dinara_mlp_predict(state["net"].value, rows, x, state["out"].ctypes.data))
        return {"predictions": state["out"]}
    _check(handle.dinara_mlp_gradients(state["net"].value, rows, x, y, state["gradients"].ctypes.data,
                                       ctypes.byref(loss)))
    return {"gradients": state["gradients"], "loss": float(loss.value)}


# ------------------------------------------------------------------ what a pass cannot do without

def _letters(case):
    """The mean letters of a pair's reference and query (a log-normal's mean, cut at the longest)."""
    mean = min(case["length"] * math.exp(case["sigma"] ** 2 / 2), float(case["longest"]))
    return (float(max(case["window"], mean)) if case["window"] else mean), mean


def work(case):
    if case["path"] == "network":
        weights = STRIDE * HIDDEN + HIDDEN * HIDDEN + 3 * HIDDEN + 1
        rows = case["rows"] * (case["epochs"] if case["op"] == "train" else 1)
        products = 1 if case["op"] == "predict" else 3
        return {"bytes": case["rows"] * (STRIDE + 1) * 4.0 + 8.0 * weights, "flops": products * 2.0 * rows * weights}
    n, m = _letters(case)
    pairs, edits = case["pairs"], m * (case["low"] + case["high"]) / 2
    # Letters as the form holds them: bytes in host memory, or packed on the device (2 bits of DNA, else a byte).
    a_letter = 1.0 if case["form"] != "resident" or case["letters"] != "dna" or case["path"] == "scoring" else 0.25
    out = 8.0 + (64.0 + 4.0 * edits if case["op"] == "alignments" else 0.0)
    if case["path"] == "scoring" or case["mode"] != "global":
        cells, ops = n * m, 10.0  # every cell may hold the best
    elif case["costs"] == "unit":
        cells, ops = m * (edits + 3), 34.0 / 64  # the narrowest band that proves the cost, 64 cells a word
    else:
        cost = 6.0 * edits
        cells, ops = m * (max(cost / 2 - 6, 0) + 3), 7.0
    return {"bytes": pairs * ((n + m) * a_letter + out), "flops": pairs * cells * ops}


# ------------------------------------------------------------------ the network's numbers in 64 bits

def exact(case, seed):
    if case["path"] != "network" or case["op"] == "train":
        return None  # alignments: whole numbers; training: the order of its shuffled batches is the library's own
    x, y = (v.double().cpu() for v in _rows(case, seed))
    w = _weights(seed).double()
    sizes = [STRIDE * HIDDEN, HIDDEN, HIDDEN * HIDDEN, HIDDEN, HIDDEN, 1]
    w1, b1, w2, b2, w3, b3 = torch.split(w, sizes)
    w1, w2 = w1.reshape(STRIDE, HIDDEN), w2.reshape(HIDDEN, HIDDEN)
    z1 = x @ w1 + b1
    a1 = z1.clamp_min(0)
    z2 = a1 @ w2 + b2
    a2 = z2.clamp_min(0)
    out = a2 @ w3 + b3
    if case["op"] == "predict":
        return {"predictions": out}
    d = 2 * (out - y) / len(y)
    dz2 = d[:, None] * w3 * (z2 > 0)
    dz1 = (dz2 @ w2.T) * (z1 > 0)
    gradients = torch.cat([(x.T @ dz1).reshape(-1), dz1.sum(0), (a1.T @ dz2).reshape(-1), dz2.sum(0), a2.T @ d,
                           d.sum().reshape(1)])
    return {"gradients": gradients, "loss": float(((out - y) ** 2).mean())}
