"""Bands wider than the first level of the one-DP-per-wavefront kernel (960 diagonals, oic_wdp.h) inside a search, where
a pair that outgrows it is run again from its start: against the oracle."""
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
