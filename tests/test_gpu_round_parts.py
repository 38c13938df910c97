"""Process_Matches in rounds (oic_rounds.h) beyond what its arrays hold at once, against the oracle: more candidate pairs
than take their rounds together (2^20), and pairs whose extensions need several fillings of the mask store; and pairs
with more extensions than the cost model expects."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


def tandem_pair(seed, unit, copies, div, err):
    """Two reads of one tandem array whose copies differ by div, with err sequencing differences."""
    rng = np.random.default_rng(seed)
    base = rng.integers(0, 4, unit)
    array = np.concatenate([np.where(rng.random(unit) < div, rng.integers(0, 4, unit), base) for _ in range(copies)])
    seqs = []
    for _ in range(2):
        u = rng.random(len(array))
        s = np.where(u < err / 2, (array + 1) % 4, array)[u < 1 - err / 2]
        seqs.append("".join("ACGT"[x] for x in s[int(rng.integers(0, unit)):]))
    return readsim.from_strings(seqs)


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


def run_both(R, minlength, partial, expected=None):
    """expected: a model that expects so many DP cells of every pair, in place of the static estimate."""
    schedule = oic.SCHED_BATCHED if expected is None else oic.SCHED_LEARNED
    eng = oic.Engine(kmer=22, maxerate=0.045, minlength=minlength, threads=1, schedule=schedule, partial=partial)
    if expected is not None:
        w = np.zeros(oic.NPARAM, np.float32)
        w[-2] = np.log1p(expected)
        eng.set_model(w, np.zeros(oic.NFEAT, np.float32), np.ones(oic.NFEAT, np.float32))
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(R, kmer=22, maxErate=0.045, minOlap=minlength, nThreads=1, ompThreads=16, partial=int(partial))
    assert res.counters["pairs"] == ref["pairs"]
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    assert list(res.stats) == list(ref["stats"])
    assert res.counters["extensions"] == ref["extensions"] and res.counters["dp_cells"] == ref["cells_used"]
    return res


@pytest.mark.parametrize("partial", [False, True])
def test_more_pairs_than_one_part(partial):
    res = run_both(array_reads(1500, 81), 40, partial)
    assert res.counters["pairs"] > 1 << 20 and len(res.records) > 1 << 20


@pytest.mark.parametrize("copies", [60, 100])
def test_store_is_emptied_when_full(copies):
    """A pair asks for at most 64 extensions a round, each with a mask of nodes / 64 words, and the store holds 4 words
    a node (65536 at least): a few hundred extensions.  Rounds that went on with a full store, until tasks without
    work had used up a place for every node, were more than (nodes - that many) / 64."""
    c = run_both(tandem_pair(75, 130, copies, 0.02, 0.012), 500, True).counters
    words, store = (c["nodes"] + 63) // 64, max(1 << 16, 4 * c["nodes"])
    assert c["pairs"] == 1 and c["extensions"] * words > 2 * store
    assert c["pp_launches"] < c["nodes"] / 128 < (c["nodes"] - store / words) / 64


@pytest.mark.parametrize("expected", [0, 1000, 100_000])
def test_used_up_prediction_does_not_add_rounds(expected):
    """Low-error pairs, of some ten extensions of several thousand cells each.  A model that expects too little holds
    back what a pair asks for until its expectation is used up, for a round or two; a round an extension from then on
    would be tens."""
    R = readsim.simulate(readsim.PRESETS["c1"].scaled(60_000, seed=82))
    few, many = run_both(R, 500, False, expected).counters, run_both(R, 500, False).counters
    assert few["learned_pairs"] == few["pairs"] and few["extensions"] > 8 * few["pairs"]
    assert few["pp_launches"] <= many["pp_launches"] + 3
