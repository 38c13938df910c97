"""The flat-row kernel (k_fwd_flat) on the tasks of small searches, which by default run one to a wavefront: reads with N
and odd lengths, fewer tasks than a wavefront has groups, pools that run out.  Against the oracle, with the packed
kernel's own cells as the proof that it ran."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu

# task order 1 and the counters keep passes of few tasks in the packed kernel; the latter is another instance of it
FORMS = [dict(fwd_lanes=4, fwd_tile=64, fwd_order=1), dict(fwd_lanes=8, fwd_tile=64, fwd_order=1),
         dict(fwd_lanes=4, fwd_tile=32, fwd_order=1), dict(fwd_lanes=8, fwd_tile=128, fwd_order=1),
         dict(fwd_lanes=4, fwd_tile=64, fwd_counters=1), dict(fwd_lanes=8, fwd_tile=64, fwd_counters=1)]


def form_id(t):
    return f"{t['fwd_lanes']}x{t['fwd_tile']}" + ("-counters" if "fwd_counters" in t else "")


def check(R, tuning, maxerate=0.045):
    eng = oic.Engine(kmer=22, maxerate=maxerate, minlength=500, threads=1, schedule=oic.SCHED_BATCHED)
    eng.set_tuning(fwd_loop=2, **tuning)
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(R, kmer=22, maxErate=maxerate, minOlap=500, nThreads=1, ompThreads=16)
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    c = res.counters
    assert list(res.stats) == list(ref["stats"])
    assert c["dp_cells"] == ref["cells_used"] and c["extensions"] == ref["extensions"]
    # the cells of a DP that outgrows the tile are those of its run at the next level
    assert c["fwd_launches"] > 0 and (c["fwd_cells"] > 0 or c["overflow_retries"] > 0)
    return c


def with_n(R, rng, every, count):
    """Every so many-th read with N at `count` places, among them its first and last base and a run of 20."""
    seqs = [R.read(i).decode() for i in range(1, R.n + 1)]
    for i in range(0, len(seqs), every):
        s = list(seqs[i])
        at = int(rng.integers(0, len(s) - 20))
        for p in [0, len(s) - 1, *range(at, at + 20), *rng.integers(0, len(s), count)]:
            s[p] = "N"
        seqs[i] = "".join(s)
    return seqs


@pytest.mark.parametrize("tuning", FORMS, ids=form_id)
@pytest.mark.parametrize("preset,genome", [("c1", 60_000), ("c3", 400_000)])
def test_reads_with_n_and_odd_lengths(preset, genome, tuning):
    rng = np.random.default_rng(96)
    R = readsim.simulate(readsim.PRESETS[preset].scaled(genome, seed=97))
    seqs = with_n(R, rng, 3, 5)
    seqs = [s[:len(s) - i % 37] for i, s in enumerate(seqs)]      # ends at every place of a word and of its 32-base group
    seqs[1] = seqs[1][:300]                                       # shorter than --minlength
    seqs.append("ACGT" * 3)                                       # and than k
    check(readsim.from_strings(seqs), tuning)


@pytest.mark.parametrize("tuning", FORMS, ids=form_id)
@pytest.mark.parametrize("reads", [2, 3, 6, 7, 17])
def test_fewer_tasks_than_groups(reads, tuning):
    """1 to 136 pairs of one locus: a pass of fewer tasks than a wavefront's 8 or 16 groups, and a little more."""
    rng = np.random.default_rng(reads)
    base = rng.integers(0, 4, 2500)
    seqs = []
    for i in range(reads):
        u = rng.random(len(base))
        s = np.where(u < 0.01, (base + 1) % 4, base)[u < 0.985]
        seqs.append("".join("ACGT"[x] for x in s[int(rng.integers(0, 400)):len(s) - int(rng.integers(0, 400))]))
    seqs = with_n(readsim.from_strings(seqs), rng, 2, 2)
    c = check(readsim.from_strings(seqs), tuning)
    assert 0 < c["pairs"] <= reads * (reads - 1)
