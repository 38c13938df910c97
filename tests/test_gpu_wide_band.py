"""Bands wider than the first level of the one-DP-per-wavefront kernel (960 diagonals, oic_wdp.h) inside a search, where
a pair that outgrows it is run again from its start, and the entry point without allocation, whose row store ends
before such a band: against the oracle and against oic_prefix_dp_batch."""
import ctypes

import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


def mutate(rng, s, rate):
    """2-bit codes with substitutions, insertions and deletions at rate / 3 each."""
    u = rng.random(len(s))
    out = []
    for x, v in zip(s, u):
        if v < rate / 3:
            out.append((x + 1 + int(rng.integers(0, 3))) % 4)
        elif v < 2 * rate / 3:
            out += [int(rng.integers(0, 4)), x]
        elif v >= rate:
            out.append(x)
    return np.array(out)


def text(s):
    return "".join("ACGT"[x] for x in s)


@pytest.mark.parametrize("schedule", [oic.SCHED_PLAIN, oic.SCHED_BATCHED], ids=["plain", "batched"])
@pytest.mark.parametrize("partial", [False, True])
def test_search_runs_wide_pairs_again(schedule, partial):
    """Reads of 33 kbp that share their first 400 bases exactly and differ by 3 % after them: the longest match is at
    one end, so the extension's right tail holds some 950 errors and, at a limit of 12 %, a band of more than 960."""
    rng = np.random.default_rng(91)
    head, base = rng.integers(0, 4, 400), rng.integers(0, 4, 32_600)
    seqs = [text(np.concatenate([head, s])) for s in (base, mutate(rng, base, 0.03), mutate(rng, base, 0.03))]
    R = readsim.from_strings(seqs + [text(base[5000:9000])])
    eng = oic.Engine(kmer=22, maxerate=0.12, minlength=500, threads=1, schedule=schedule, partial=partial)
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(R, kmer=22, maxErate=0.12, minOlap=500, nThreads=1, ompThreads=8, partial=int(partial))
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) > 0 and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    assert list(res.stats) == list(ref["stats"])
    c = res.counters
    assert c["extensions"] == ref["extensions"] and c["dp_cells"] == ref["cells_used"]
    assert c["overflow_retries"] >= 2       # base with each of the other two, at the least


@pytest.mark.parametrize("limit", [1, 479, 480, 700, 1021])
def test_noalloc_at_limits_around_the_first_level(limit):
    """Tasks that the store of 131072 cells holds (at most (e + 1)^2 of them for e errors) beside ones that it does not:
    a band past 960 has kept more cells than that."""
    rng = np.random.default_rng(92)
    seqs, tasks = [], []
    for length in (40, 3000, 9000, 26_000):
        a = rng.integers(0, 4, length)
        seqs += sorted((text(a), text(mutate(rng, a, 0.03))), key=len)
        m, n, i = len(seqs[-2]), len(seqs[-1]), len(seqs) - 1
        tasks += [(i, i + 1, 0, 0, 0, 0, m, n, limit, 0), (i, i + 1, 0, 0, m - 1, n - 1, m, n, limit, 1)]
    eng = oic.Engine(kmer=22, maxerate=0.12)
    eng.load_reads(readsim.from_strings(seqs + ["ACGT" * 10_000]))
    tasks = np.array(tasks, oic.DP_TASK)
    want, wdelta = eng.prefix_dp(tasks, delta_stride=1024)
    assert (want["status"] == 0).all()
    res, delta = np.zeros(len(tasks), oic.DP_RESULT), np.full((len(tasks), 1024), -7, np.int32)
    rc = oic.lib().oic_prefix_dp_batch_noalloc(eng._ctx, tasks.ctypes.data, len(tasks), res.ctypes.data, delta.ctypes.data,
                                               ctypes.c_uint32(1024))
    assert rc == oic.OIC_OK
    fits = np.arange(len(tasks)) < (len(tasks) if limit == 1 else 6)
    assert (res["status"][fits] == 0).all() and (res["status"][~fits] == oic.OIC_ECAPACITY).all()
    assert np.array_equal(res[fits], want[fits])
    for k in np.flatnonzero(fits):
        d = int(want["delta_len"][k])
        assert np.array_equal(delta[k][:d], wdelta[k][:d]) and (delta[k][d:] == 0).all()
