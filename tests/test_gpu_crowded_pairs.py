"""Match lists of pairs with few hits in all but many at one S offset, against the oracle: past the 64 that the
wavefront level of such pairs holds, and past the 512 of the last wavefront level."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies,offsets", [(60, 6), (64, 6), (65, 6), (70, 20), (129, 9), (300, 5), (512, 3), (513, 3), (600, 2)])
def test_crowded_offsets_of_small_pairs(copies, offsets):
    rng = np.random.default_rng(copies)

    def rand(n):
        return "".join(rng.choice(list("ACGT"), n))

    unit, left, right = rand(53), rand(400), rand(400)
    seqs = [left + unit[:21 + offsets] + rand(30) + right, left + rand(30) + unit * copies + right]
    R = readsim.from_strings(seqs + [left[200:] + right + rand(50)])
    eng = oic.Engine(kmer=22, maxerate=0.045, minlength=40, threads=1, schedule=oic.SCHED_BATCHED)
    eng.set_tuning(list_wave_min_hits=4096)           # all pairs are pairs of few hits
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(R, kmer=22, maxErate=0.045, minOlap=40, nThreads=1, ompThreads=8)
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    c = res.counters
    assert list(res.stats) == list(ref["stats"]) and c["hits"] == ref["hits"]
    assert c["extensions"] == ref["extensions"] and c["dp_cells"] == ref["cells_used"]
    assert c["list_wave_pairs"] == 0
    assert (c["list_second_level"] > 0) == (copies > 64) and (c["list_handed_back"] > 0) == (copies > 512)
