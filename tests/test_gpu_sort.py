"""The radix sort under the k-mer table and the hit grouping, through whole searches against the oracle: positions
around a tile's 8192 keys, read counts whose bits take 8, 9, 10 and 11-bit digits in one pass and two, and reads
with N, whose invalid windows sort last."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


def rand_seq(rng, n):
    return "".join(rng.choice(list("ACGT"), n))


def check(R):
    eng = oic.Engine(kmer=22, maxerate=0.045, minlength=40, threads=1, schedule=oic.SCHED_BATCHED)
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(R, kmer=22, maxErate=0.045, minOlap=40, nThreads=1, ompThreads=8)
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    assert res.counters["hits"] == ref["hits"] and res.counters["pairs"] == ref["pairs"]
    assert res.counters["dp_cells"] == ref["cells_used"] and res.counters["extensions"] == ref["extensions"]
    return res.counters


@pytest.mark.parametrize("positions", [1, 2, 8191, 8192, 8193, 16384, 8 * 8192, 8 * 8192 + 1])
def test_positions_around_a_tile(positions):
    rng = np.random.default_rng(positions)
    each = min(positions, 4096)
    genome = rand_seq(rng, 6000)
    seqs, left = [], positions
    while left:
        n = min(each, left) + 21                  # a read of n bases holds n - 21 k-mers
        n = max(n, 40) if left < 19 else n
        at = int(rng.integers(0, len(genome) - n + 1))
        seqs.append(genome[at:at + n])
        left -= min(each, left)
    check(readsim.from_strings(seqs))


@pytest.mark.parametrize("reads", [200, 256, 257, 512, 513, 1025, 2047, 2049, 4100])
def test_digit_widths(reads):
    rng = np.random.default_rng(reads)
    genome = rand_seq(rng, 20 * reads)
    seqs = []
    for _ in range(reads):
        n = int(rng.integers(45, 120))
        at = int(rng.integers(0, len(genome) - n + 1))
        s = genome[at:at + n]
        if rng.random() < 0.1:
            p = int(rng.integers(0, n))
            s = s[:p] + "N" + s[p + 1:]
        seqs.append(s)
    assert check(readsim.from_strings(seqs))["hits"] > 0
