"""The one-DP-per-wavefront kernel (oic_wdp.h) against the oracle where its parts meet: slides that end around
its 48-base windows and 1024-base steps, error limits around the 64 rows whose limits it holds and the 31 a
traceback walks at once, bands around its first level's width, deltas of hundreds of entries."""
import numpy as np
import pytest

from canu_amd import oic, readsim
from oracle import oracle

pytestmark = pytest.mark.gpu


def rand_seq(rng, n):
    return "".join(rng.choice(list("ACGT"), n))


def mutate(rng, s, rate):
    u = rng.random(len(s))
    out = []
    for ch, x in zip(s, u):
        if x < rate / 3:
            out.append("ACGT"[("ACGT".index(ch) + 1 + int(rng.integers(0, 3))) % 4])
        elif x >= 2 * rate / 3 and x < rate:
            out.append(rand_seq(rng, 1) + ch)
        elif x >= rate:
            out.append(ch)
    return "".join(out)


def check(pairs, rate, limits):
    """forward and reverse on each (a, b), every error limit, against the oracle: results, deltas and cells."""
    seqs, tasks = [], []
    for a, b in pairs:
        if len(a) > len(b):
            a, b = b, a
        seqs += [a, b]
        m, n, i = len(a), len(b), len(seqs) - 1
        for lim in limits:
            tasks += [(i, i + 1, 0, 0, 0, 0, m, n, lim, 0), (i, i + 1, 0, 0, m - 1, n - 1, m, n, lim, 1)]
    # the engine sizes its row store for the error limit of the longest read: one that no task uses
    R = readsim.from_strings(seqs + ["ACGT" * 10_000])
    eng = oic.Engine(kmer=22, maxerate=rate)
    eng.load_reads(R)
    t = np.array(tasks, oic.DP_TASK)
    res, delta = eng.prefix_dp(t, delta_stride=4096)
    od = oracle.OracleDP(rate)
    od.reset_counters()
    for k, tk in enumerate(t):
        A, B, r = seqs[tk["a_id"] - 1].lower().encode(), seqs[tk["b_id"] - 1].lower().encode(), res[k]
        assert r["status"] == 0, k
        if tk["dir"] == 0:
            e, ae, te, mte, d = od.forward(A, B, int(tk["error_limit"]))
        else:
            e, ae, te, lo, mte, d = od.reverse(A, B, int(tk["error_limit"]))
            assert r["leftover"] == lo, k
        assert (r["errors"], r["a_end"], r["t_end"], bool(r["match_to_end"])) == (e, ae, te, mte), (k, tk)
        assert r["delta_len"] == len(d) and np.array_equal(delta[k][:len(d)], d), k
    assert int(res["cells"].sum()) == od.counters()["cells"]
    return res


@pytest.mark.parametrize("with_n", [False, True])
@pytest.mark.parametrize("run", [1, 15, 16, 47, 48, 49, 63, 64, 96, 112, 1023, 1024, 1025, 1071, 1072, 1073, 2200])
def test_slides_of_every_step(run, with_n):
    rng = np.random.default_rng(run)
    pairs = []
    for gap in (0, 1, 3):
        # runs of that many equal bases between a substitution, an insertion or nothing, the last one to the end
        parts = [rand_seq(rng, run) for _ in range(4)]
        other = ["A" if p[-1] != "A" else "C" for p in parts]
        a, b = "".join(parts), "".join(p[:-1] + o for p, o in zip(parts, other)) + rand_seq(rng, gap)
        if with_n:
            k = len(a) // 2
            a = a[:k] + "N" + a[k + 1:]
        pairs += [(a, b), (a, parts[0] + "G" + "".join(parts[1:])), (a, a + rand_seq(rng, gap))]
    check(pairs, 0.045, [3, 8])


@pytest.mark.parametrize("limit", [0, 1, 30, 31, 32, 33, 62, 63, 64, 65, 128])
def test_error_limits_around_the_row_blocks(limit):
    rng = np.random.default_rng(100 + limit)
    pairs = [(a, mutate(rng, a, r)) for r in (0.02, 0.04) for a in (rand_seq(rng, int(n)) for n in rng.integers(300, 4000, 6))]
    check(pairs, 0.045, [limit])


@pytest.mark.parametrize("length", [9000, 14000, 26000])
def test_bands_around_the_first_level(length):
    """3 % difference at a 12 % limit: bands grow by about 1.5 diagonals a row, past 960 at 14 kbp and more."""
    rng = np.random.default_rng(length)
    pairs = [(a, mutate(rng, a, 0.03)) for a in (rand_seq(rng, length) for _ in range(3))]
    res = check(pairs, 0.12, [900])
    assert res["delta_len"].max() > 100
