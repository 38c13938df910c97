"""Work counters whose meaning depends on the path a call takes: the packed forward kernel's launches, bands re-run at
every level, and the extensions run ahead of Process_Matches."""
import numpy as np
import pytest

from canu_amd import oic, readsim

pytestmark = pytest.mark.gpu


def run(R, schedule=oic.SCHED_BATCHED, tuning=None, **opt):
    eng = oic.Engine(**{**dict(kmer=22, maxerate=0.045, minlength=500, threads=1, schedule=schedule), **opt})
    if tuning:
        eng.set_tuning(**tuning)
    eng.load_reads(R)
    return eng.run().counters


@pytest.mark.parametrize("graph", [1, 0])
def test_packed_launches_are_those_that_ran(graph):
    """Few forward DPs run one to a wavefront, and the packed kernel's launches for them return at once."""
    R = readsim.simulate(readsim.PRESETS["c1"].scaled(60_000, seed=93))
    few = run(R, tuning=dict(fwd_graph=graph))
    assert few["fwd_launches"] == 0 and few["fwd_cells"] == 0 and few["spec_cells"] > few["pp_cells"] > 0
    packed = run(R, tuning=dict(fwd_order=1))           # all of them in the packed kernel
    assert 1 <= packed["fwd_launches"] <= 2 and packed["fwd_cells"] > 0
    assert packed["dp_cells"] == few["dp_cells"]


def test_bands_rerun_from_every_level():
    """Two reads of 33 kbp that differ by 3 % behind a common start: the forward DP outgrows the first level, 960
    diagonals, of the one-per-wavefront kernel, which here takes the tasks first."""
    rng = np.random.default_rng(94)
    head, base = rng.integers(0, 4, 400), rng.integers(0, 4, 32_600)
    u = rng.random(len(base))
    other = np.where(u < 0.01, (base + 1) % 4, base)[u < 0.98]
    other = np.insert(other, rng.integers(0, len(other), 326), 0)
    R = readsim.from_strings(["".join("ACGT"[x] for x in np.concatenate([head, s])) for s in (base, other)])
    c = run(R, maxerate=0.12)
    assert c["pairs"] == 1 and c["fwd_launches"] == 0
    assert c["overflow_retries"] >= 2                   # the probe's forward DP, then the pair's extension


def test_tasks_run_ahead_are_real_ones():
    """One tandem pair under -partial: every extension that runs has one or two DPs, and no forward pass adds any."""
    rng = np.random.default_rng(95)
    unit = rng.integers(0, 4, 130)
    array = np.concatenate([np.where(rng.random(130) < 0.02, rng.integers(0, 4, 130), unit) for _ in range(60)])
    seqs = []
    for _ in range(2):
        u = rng.random(len(array))
        seqs.append("".join("ACGT"[x] for x in np.where(u < 0.006, (array + 1) % 4, array)[u < 0.994]))
    c = run(readsim.from_strings(seqs), partial=True)
    assert c["pairs"] == 1 and c["extensions"] > 500
    assert c["extensions"] <= c["spec_tasks"] <= c["dp_calls"] <= 2 * c["spec_tasks"]
