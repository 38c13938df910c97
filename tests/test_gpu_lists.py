"""The wavefront list builders (k_build_lists_wave) against the oracle where their parts meet: pairs whose hits
end around the 64-hit block and the 128-hit window, runs broken at every place of a block, offsets of several
hits between blocks of single ones, and pairs long enough to be built in parts.  Process_Matches picks nodes in
list order, so records, extensions and DP cells depend on it."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


def rand_seq(rng, n):
    return "".join(rng.choice(list("ACGT"), n))


def other_base(ch):
    return "ACGT"["CATG".index(ch)]


def check(R, min_hits, **opt):
    okw = {("minOlap" if k == "minlength" else k): int(v) for k, v in opt.items()}
    eng = oic.Engine(**{**dict(kmer=22, maxerate=0.045, minlength=40, threads=1, schedule=oic.SCHED_BATCHED), **opt})
    if min_hits is not None:
        eng.set_tuning(list_wave_min_hits=min_hits)
    eng.load_reads(R)
    res = eng.run()
    ref = oracle.run(R, **{**dict(kmer=22, maxErate=0.045, minOlap=40, nThreads=1, ompThreads=8), **okw})
    a, b = oic.sort_records(res.records), oracle.sort_records(ref["records"])
    assert len(a) == len(b) and all(np.array_equal(a[f], b[f]) for f in ("a_iid", "b_iid", "w0", "w1"))
    assert list(res.stats) == list(ref["stats"])
    assert res.counters["hits"] == ref["hits"] and res.counters["pairs"] == ref["pairs"]
    assert res.counters["dp_cells"] == ref["cells_used"] and res.counters["extensions"] == ref["extensions"]
    return res.counters


@pytest.mark.parametrize("min_hits", [None, 0])
@pytest.mark.parametrize("hits", [1, 2, 62, 63, 64, 65, 66, 126, 127, 128, 129, 130, 192, 193, 257])
def test_blocks_of_single_hits(hits, min_hits):
    rng = np.random.default_rng(hits)
    seqs = []
    for breaks in (0, 1, 2, 5):
        a = rand_seq(rng, hits + 21)
        b = list(a)
        for p in rng.integers(0, len(a), breaks):
            b[p] = other_base(b[p])                 # 22 offsets without a hit
        cut = int(rng.integers(0, len(a)))
        seqs += [a + rand_seq(rng, 60), "".join(b) + rand_seq(rng, 60),
                 a[:cut] + rand_seq(rng, int(rng.integers(1, 4))) + a[cut:]]   # another diagonal from there on
    c = check(readsim.from_strings(seqs), min_hits)
    assert c["hits"] > 0


@pytest.mark.parametrize("min_hits", [None, 0])
@pytest.mark.parametrize("gap", [0, 20, 41, 42, 43, 64, 85])
def test_offsets_of_several_hits_between_blocks(gap, min_hits):
    """A unit that T holds three times: its offsets hold three hits each, those around them one."""
    rng = np.random.default_rng(500 + gap)
    unit, left, right = rand_seq(rng, 60), rand_seq(rng, 90), rand_seq(rng, 110)
    s = left + unit + right
    t = left + unit + rand_seq(rng, gap) + unit + rand_seq(rng, gap) + unit + right
    u = left + unit + other_base(unit[0]) + unit[1:] + right
    check(readsim.from_strings([s, t, u, t[10:]]), min_hits)


@pytest.mark.parametrize("min_hits", [None, 0, 16384])
@pytest.mark.parametrize("copies,errors", [(20, 0), (20, 4), (60, 30), (150, 12), (560, 3)])
def test_long_pairs_in_parts(copies, errors, min_hits):
    """Tandem units: an S of 24 copies with errors (gaps in its offsets) against a T of many (that many hits at
    an offset: below and above 64, 128 and 512), and a plain overlap of 9 kbp, with one gap."""
    rng = np.random.default_rng(900 + copies + errors)
    unit, left, right = rand_seq(rng, 33), rand_seq(rng, 300), rand_seq(rng, 300)
    s = list(left + unit * 24 + right)
    for p in rng.integers(0, len(s), errors):
        s[p] = other_base(s[p])
    t = left + unit * copies + right
    plain = rand_seq(rng, 9000)
    spot = 4500 + int(rng.integers(0, 300))
    R = readsim.from_strings(["".join(s), t, plain, plain[:spot] + other_base(plain[spot]) + plain[spot + 1:]])
    c = check(R, min_hits)
    assert c["hits"] > 8192 + 8900
    if min_hits == 0:
        assert c["list_wave_pairs"] == c["pairs"]
        assert (c["list_second_level"] > 0) == (copies > 128) and (c["list_handed_back"] > 0) == (copies > 512)
