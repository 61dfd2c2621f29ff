"""The C ABI's threading contract: the library keeps no state between calls that one caller's batch could see from
another's, and may be called from many host threads at once (reference c/dinara.h:14-16; its pthreads batches,
c/dinara.mojo:822-990). Several threads call dinara_alignments / dinara_distances at the same time, on different
batches and costs, and each must get exactly what the same call made alone returns.
"""

import ctypes
import threading

import pytest

from dinara_align import _lib, synthetic

pytestmark = pytest.mark.gpu


def alignments(refs, qrys, costs, threads):
    h = _lib.lib()
    R, Q = _lib.Texts(refs), _lib.Texts(qrys)
    found = (_lib.CAlignment * len(refs))()
    statuses = (ctypes.c_int64 * len(refs))()
    code = h.dinara_alignments(len(refs), *R.args(), *Q.args(), ctypes.byref(costs) if costs else None, None, None,
                               threads, found, statuses)
    out = []
    for i in range(len(refs)):
        if statuses[i] == 0:
            out.append((found[i].cost, ctypes.string_at(found[i].cigar, found[i].cigar_length)))
            h.dinara_free(found[i].cigar)
        else:
            out.append(statuses[i])
    return code, out


def distances(refs, qrys, costs, threads):
    h = _lib.lib()
    R, Q = _lib.Texts(refs), _lib.Texts(qrys)
    out = (ctypes.c_int64 * len(refs))()
    code = h.dinara_distances(len(refs), *R.args(), *Q.args(), ctypes.byref(costs) if costs else None, None, None,
                              threads, out)
    return code, list(out)


def test_concurrent_calls_from_host_threads_match_calls_alone():
    affine = _lib.CCosts(4, 6, 2, -1, 0, 0, 0, -1, 0)
    jobs = []
    for t in range(6):
        if t % 3 == 0:
            refs, qrys = synthetic.affine_reads(1500, seed=300 + t)
            jobs.append((alignments, refs, qrys, affine))
        elif t % 3 == 1:
            refs, qrys = synthetic.uneven(800, seed=300 + t, clip=(20, 2500))
            jobs.append((alignments, refs, qrys, None))
        else:
            refs, qrys = synthetic.uneven(1200, seed=300 + t, clip=(20, 2500))
            jobs.append((distances, refs, qrys, affine))
    alone = [fn(refs, qrys, costs, 2) for fn, refs, qrys, costs in jobs]
    assert all(code == 0 for code, _ in alone)
    print(f"[threads] {len(jobs)} batches alone done", flush=True)
    together = [None] * len(jobs)
    start = threading.Barrier(len(jobs))

    def worker(i):
        fn, refs, qrys, costs = jobs[i]
        start.wait()
        together[i] = fn(refs, qrys, costs, 2)

    pool = [threading.Thread(target=worker, args=(i,)) for i in range(len(jobs))]
    for t in pool:
        t.start()
    for t in pool:
        t.join(timeout=300)
    assert not any(t.is_alive() for t in pool)
    print(f"[threads] {len(jobs)} batches at once done", flush=True)
    for i, (want, got) in enumerate(zip(alone, together)):
        assert got == want, i


def test_batches_held_together_and_freed_out_of_order():
    # Resident batches whose buffers lie in blocks a context hands out and takes back: more at once than it hands out
    # (64 small, 4 large), run again, freed out of order, their blocks taken by batches of other sizes and costs, and a
    # small batch's results in one copy (up to 256 pairs) or several. Each against the same call made alone.
    h = _lib.lib()
    affine = _lib.CCosts(4, 6, 2, -1, 0, 0, 0, -1, 0)
    calls = [(*synthetic.affine_reads(pairs, seed=700 + k, length=length), costs)
             for k, (pairs, length, costs) in enumerate([(2, 60, None), (256, 90, affine), (257, 60, None),
                                                         (30, 400, affine), (6000, 100, affine)])]
    alone = [alignments(refs, qrys, costs, 2)[1] for refs, qrys, costs in calls]
    texts = [(_lib.Texts(refs), _lib.Texts(qrys)) for refs, qrys, _ in calls]

    def make(k):
        status = ctypes.c_int64(0)
        costs = calls[k][2]
        batch = h.dinara_batch_new(0, _lib.BATCH_ALIGNMENTS, len(calls[k][0]), *texts[k][0].args(),
                                   *texts[k][1].args(), ctypes.byref(costs) if costs else None, None, None, 2,
                                   ctypes.byref(status))
        assert batch, status.value
        return k, batch

    def check(held):
        k, batch = held
        found = (_lib.CAlignment * len(calls[k][0]))()
        statuses = (ctypes.c_int64 * len(calls[k][0]))()
        assert h.dinara_batch_run(batch) == 0 and h.dinara_batch_alignments(batch, found, statuses) == 0
        assert not any(statuses)
        assert [(f.cost, ctypes.string_at(f.cigar, f.cigar_length)) for f in found] == alone[k], k
        for f in found:
            h.dinara_free(f.cigar)

    held = [make(k % 4) for k in range(72)] + [make(4) for _ in range(6)]
    for batch in held:
        check(batch)
    for at in list(range(0, len(held), 2)) + list(range(len(held) - 1, 0, -2)):
        check(held[at])
        h.dinara_batch_free(held[at][1])
        again = make((at + 1) % 5)
        check(again)
        h.dinara_batch_free(again[1])
