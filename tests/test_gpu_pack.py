"""Packing of reads on the device (both strands, N masks) through whole jobs against the oracle: read lengths around
the 16- and 32-base words, lower case, and N at the words' ends and the reads'.  Any other letter is N to the engine;
the oracle compares letters, so it gets N in their place."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["plain", "lower", "N", "other"])
@pytest.mark.parametrize("length", [40, 47, 48, 49, 63, 64, 65, 95, 96, 97, 127, 128, 129, 271])
def test_words_and_ends(length, kind):
    rng = np.random.default_rng(1000 + length)
    comp = str.maketrans("ACGTacgt", "TGCAtgca")
    genome = "".join(rng.choice(list("ACGT"), 2 * length))
    seqs = []
    for at in list(range(0, length, max(1, length // 12))) + [length]:
        for flip in (False, True):
            s = genome[at:at + length]
            s = s.translate(comp)[::-1] if flip else s
            if kind == "lower":
                s = "".join(c.lower() if rng.random() < 0.5 else c for c in s)
            elif kind != "plain" and rng.random() < 0.6:
                p = int(rng.choice([0, 1, 15, 16, 31, 32, 33, length - 17, length - 16, length - 2, length - 1]))
                s = s[:p] + ("N" if kind == "N" else rng.choice(list("n-RXa@"))) + s[p + 1:]
            seqs.append(s)
    R = readsim.from_strings(seqs)
    eng = oic.Engine(kmer=16, maxerate=0.045, minlength=30, threads=1, schedule=oic.SCHED_BATCHED)
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(readsim.from_strings(["".join(c if c in "ACGTacgt" else "N" for c in s) for s in seqs]), kmer=16, maxErate=0.045, minOlap=30, nThreads=1, ompThreads=8)
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    assert list(res.stats) == list(ref["stats"])
    assert res.counters["hits"] == ref["hits"] > 0 and res.counters["dp_cells"] == ref["cells_used"]
