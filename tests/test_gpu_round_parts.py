"""Process_Matches in rounds over more candidate pairs than take their rounds together (2^20): reads of one short
tandem array, every pair a candidate with several match nodes, against the oracle."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


def array_reads(n, seed):
    """Reads of 120 to 126 bases of four 33-base units, each with a unique base changed in half of them."""
    rng = np.random.default_rng(seed)
    unit = rng.integers(0, 4, 33)
    seqs = []
    for i in range(n):
        s = np.tile(unit, 4)[:120 + i % 7]
        if i % 2:
            p = int(rng.integers(0, len(s)))
            s[p] = (s[p] + 1) % 4
        seqs.append("".join("ACGT"[x] for x in s))
    return readsim.from_strings(seqs)


@pytest.mark.parametrize("partial", [False, True])
def test_more_pairs_than_one_part(partial):
    R = array_reads(1500, 81)
    eng = oic.Engine(kmer=22, maxerate=0.045, minlength=40, threads=1, schedule=oic.SCHED_BATCHED, partial=partial)
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(R, kmer=22, maxErate=0.045, minOlap=40, nThreads=1, ompThreads=16, partial=int(partial))
    assert res.counters["pairs"] == ref["pairs"] > 1 << 20
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) > 1 << 20 and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    assert list(res.stats) == list(ref["stats"])
    assert res.counters["extensions"] == ref["extensions"] and res.counters["dp_cells"] == ref["cells_used"]
