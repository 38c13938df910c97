"""Process_Matches in rounds (oic_rounds.h) against the oracle: pairs with few and many match nodes, every option
that changes what an extension removes or keeps, more nodes than the rounds' mask store holds (the pairs left
open then run one to a wavefront), and the cost model's limit on what a pair asks for."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


def tandem(seed, unit, copies, div, reads, err):
    """Reads of one tandem array whose copies differ by div, with err sequencing differences."""
    rng = np.random.default_rng(seed)
    base = rng.integers(0, 4, unit)
    array = np.concatenate([np.where(rng.random(unit) < div, rng.integers(0, 4, unit), base) for _ in range(copies)])
    seqs = []
    for _ in range(reads):
        s = array.copy()
        u = rng.random(len(s))
        s = np.where(u < err / 2, (s + 1) % 4, s)
        s = s[u < 1 - err / 2]
        cut = int(rng.integers(0, unit))
        seqs.append("".join("ACGT"[x] for x in s[cut:]))
    return readsim.from_strings(seqs)


def run_both(R, schedule, model=False, **opt):
    ekw, okw = dict(kmer=22, maxerate=0.045, minlength=500, threads=1), dict(kmer=22, maxErate=0.045, minOlap=500, nThreads=1, ompThreads=16)
    for k, v in opt.items():
        ekw[k] = v
        okw[k] = int(v)
    eng = oic.Engine(schedule=schedule, **ekw)
    if model:
        # a model that expects exp(7) cells of every pair: few extensions each
        w = np.zeros(oic.NPARAM, np.float32)
        w[-2] = 7.0
        eng.set_model(w, np.zeros(oic.NFEAT, np.float32), np.ones(oic.NFEAT, np.float32))
    eng.load_reads(R)
    res, ref = eng.run(), oracle.run(R, **okw)
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    assert list(res.stats) == list(ref["stats"])
    assert res.counters["dp_cells"] == ref["cells_used"] and res.counters["extensions"] == ref["extensions"]
    return res.counters


@pytest.mark.parametrize("opt", [dict(), dict(unique=False), dict(partial=True), dict(partial=True, unique=False), dict(hopeless=False)],
                         ids=lambda o: "-".join(f"{k}{int(v)}" for k, v in o.items()) or "default")
def test_low_error_reads(opt):
    c = run_both(readsim.simulate(readsim.PRESETS["c1"].scaled(60_000, seed=71)), oic.SCHED_BATCHED, **opt)
    assert c["pp_launches"] > 2 and c["extensions"] > 1000


@pytest.mark.parametrize("partial", [False, True])
def test_tandem_pairs_with_many_nodes(partial):
    c = run_both(tandem(72, 130, 30, 0.02, 6, 0.01), oic.SCHED_BATCHED, partial=partial)
    assert c["nodes"] > 10 * 64 * c["pairs"]      # masks of many words


def test_pairs_beyond_the_mask_store():
    c = run_both(tandem(73, 130, 44, 0.02, 2, 0.012), oic.SCHED_BATCHED, partial=True)
    words = (c["nodes"] // c["pairs"] + 63) // 64
    assert c["extensions"] * words > 1 << 16       # more than the store of a batch of so few nodes


def test_model_limits_what_a_pair_asks_for():
    R = readsim.simulate(readsim.PRESETS["c1"].scaled(60_000, seed=74))
    few, many = run_both(R, oic.SCHED_LEARNED, model=True), run_both(R, oic.SCHED_BATCHED)
    assert few["spec_tasks"] < many["spec_tasks"]
