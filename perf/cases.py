"""Performance cases of the overlapInCore engine: what its callers run, through canu_amd.oic.

Kinds of work:

  job     a whole overlapInCore call on an engine in hand: host reads in (load_reads), the hash-block loop
          over them and the overlap records out (run), with the command line's schedule;
  search  one batch of ref reads against an index that is already built (a long run's repeated step);
  extend  Extend_Alignment on seeds of true overlaps, deltas out;
  dp      prefixEditDistance::forward and ::reverse on explicit windows, deltas out;
  dp0     the same through the entry point that allocates nothing;
  train   the learned cost model: training on traces, then its predictions on others.

Reads come from the repository's own generators (canu_amd.readsim), scaled to smaller genomes with the coverage,
read lengths, error rates and repeat mix of the workload:

  c1  15x, 8 kbp, 1.5 % errors per read: low-error reads, most candidate pairs overlap;
  c2  30x, 12 kbp, 4 % errors per read, no repeats: pairs differ by more than --maxerate;
  c3  c2 with 25 % interspersed repeats and satellite arrays;
  c5  30x, 18 kbp, 0.2 % errors, homopolymer-compressed, the repeats of c3; --maxerate 0.01.
"""
import ctypes
import math

import numpy as np

from canu_amd import oic, readsim

OPTIONS = {
    "c1": dict(kmer=22, maxerate=0.045, minlength=500, hashbits=23, hashload=0.8, hashdatalen=200_000_000),
    "c2": dict(kmer=22, maxerate=0.045, minlength=500, hashbits=26, hashload=0.8, hashdatalen=2_000_000_000),
    "c3": dict(kmer=22, maxerate=0.045, minlength=500, hashbits=26, hashload=0.8, hashdatalen=2_000_000_000),
    "c5": dict(kmer=22, maxerate=0.01, minlength=1000, hashbits=27, hashload=0.8, hashdatalen=4_000_000_000),
}
MAX_RECORDS = 1 << 18     # rows of a job's or search's output buffer
SCHEDULES = {"plain": oic.SCHED_PLAIN, "batched": oic.SCHED_BATCHED, "learned": oic.SCHED_LEARNED}

# DP cells that Process_Matches consumes per base of a ref read searched against every later read of the set, as
# the engine counts them at the listed sizes.  They scale the work() of a case; nothing else reads them.
CELLS = {"c1": 360.0, "c2": 430.0, "c3": 1000.0, "c5": 120.0}


def listed():
    return [
        # the smallest job: one short contig's reads; launches, synchronisations and allocations count
        dict(name="job small", kind="job", preset="c1", genome=20_000, schedule="learned", partial=False, last_ref=0),
        # an ordinary low-error job: index, seeds, dovetail extensions with deltas, records
        dict(name="job low-error", kind="job", preset="c1", genome=400_000, schedule="learned", partial=False, last_ref=0),
        # overlaps for trimming (-partial): every extension keeps its deltas, no forward DP runs ahead
        dict(name="job trimming", kind="job", preset="c1", genome=80_000, schedule="learned", partial=True, last_ref=0),
        # one rectangle of a large assembly: a large hash block, few ref reads; loading and indexing count
        dict(name="job hash block", kind="job", preset="c2", genome=5_000_000, schedule="learned", partial=False, last_ref=25),
        # noisy reads without repeats: most extensions end at a branch point
        dict(name="search noisy", kind="search", preset="c2", genome=4_000_000, schedule="batched", refs=1500),
        # the same reads with the engine's default schedule, one candidate pair per wavefront
        dict(name="search default", kind="search", preset="c2", genome=1_000_000, schedule="plain", refs=200),
        # repeat families and satellites: crowded match lists, many short extensions
        dict(name="search repeats", kind="search", preset="c3", genome=8_000_000, schedule="batched", refs=400),
        # compressed HiFi-like reads: long exact slides, many true overlaps
        dict(name="search hifi", kind="search", preset="c5", genome=6_000_000, schedule="batched", refs=150),
        # seed extensions of a consumer that keeps its own seeds (both directions, deltas merged)
        dict(name="extend", kind="extend", tasks=600, length=8000, rate=0.03, maxerate=0.045),
        # prefix DPs on long windows at up to the error limit
        dict(name="dp long", kind="dp", tasks=400, length=12000, rate=0.06, maxerate=0.045),
        # a few short DPs from a serving loop
        dict(name="dp small", kind="dp0", tasks=12, length=600, rate=0.03, maxerate=0.045),
        # the cost model of the learned schedule
        dict(name="train", kind="train", samples=60_000, batch=4096, epochs=2),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["job", "job", "search", "search", "search", "extend", "dp", "dp0", "train"])
    if kind == "job":
        preset = rng.choice(["c1", "c1", "c2", "c3"])
        if preset == "c1":
            partial = rng.random() < 0.25
            return dict(kind=kind, preset=preset, genome=_log_uniform(rng, 10_000, 80_000 if partial else 400_000),
                        schedule="learned", partial=partial, last_ref=0)
        return dict(kind=kind, preset=preset, genome=_log_uniform(rng, 100_000, 2_000_000), schedule="learned", partial=False,
                    last_ref=_log_uniform(rng, 2, 25))
    if kind == "search":
        preset, genome, refs = rng.choice([("c1", 300_000, 250), ("c2", 2_000_000, 1500), ("c3", 4_000_000, 300), ("c5", 3_000_000, 120)])
        schedule = "plain" if preset in ("c1", "c2") and rng.random() < 0.25 else "batched"
        if schedule == "plain":
            genome, refs = genome // 2, refs // 5
        return dict(kind=kind, preset=preset, genome=_log_uniform(rng, genome // 8, genome), schedule=schedule,
                    refs=_log_uniform(rng, max(3, refs // 20), refs))
    if kind == "train":
        return dict(kind=kind, samples=_log_uniform(rng, 3_000, 60_000), batch=rng.choice([1000, 2048, 4096]), epochs=rng.randint(1, 2))
    most, longest = {"extend": (600, 8000), "dp": (400, 12000), "dp0": (64, 2000)}[kind]
    maxerate = rng.choice([0.045, 0.045, 0.12, 0.01])
    return dict(kind=kind, tasks=_log_uniform(rng, 4, most), length=_log_uniform(rng, 200, longest),
                rate=round(maxerate * rng.uniform(0.2, 1.3), 4), maxerate=maxerate)


def _mutate(rng, s, rate):
    """s with substitutions, insertions and deletions, each at rate / 3 per base."""
    u = rng.random(len(s))
    out = s.copy()
    sub = u < rate / 3
    out[sub] = (out[sub] + rng.integers(1, 4, int(sub.sum()), dtype=np.uint8)) & 3
    times = np.ones(len(s), np.int64)
    times[(u >= rate / 3) & (u < 2 * rate / 3)] = 0
    ins = (u >= 2 * rate / 3) & (u < rate)
    times[ins] = 2
    first = np.cumsum(times) - times
    out = np.repeat(out, times)
    out[first[ins]] = rng.integers(0, 4, int(ins.sum()), dtype=np.uint8)
    return out


def _read_set(seqs):
    """A 1-based readsim.Reads from 2-bit code arrays."""
    text = np.frombuffer(b"ACGT", np.uint8)
    n = len(seqs)
    length = np.zeros(n + 1, np.uint32)
    length[1:] = [len(s) for s in seqs]
    start = np.zeros(n + 1, np.uint64)
    start[1:] = np.cumsum(length.astype(np.uint64) + 1)[:-1]
    bases = np.zeros(int(length.sum()) + n, np.uint8)
    for i, s in enumerate(seqs):
        b = int(start[i + 1])
        bases[b:b + len(s)] = text[s]
    return readsim.Reads(bases, start, length, np.zeros(n + 1, np.uint64), np.zeros(n + 1, np.uint8), 0)


def _lengths(rng, n, mean):
    """Lognormal read lengths around mean, as the generators draw them."""
    sigma = 0.4
    return np.clip(rng.lognormal(math.log(mean) - sigma * sigma / 2, sigma, n), 60, 4 * mean).astype(np.int64)


def _prepare_extend(case, rng):
    seqs, tasks = [], []
    for length in _lengths(rng, case["tasks"], case["length"]):
        # an overlap of two reads around an exact seed: S starts inside T or T inside S, and one ends first
        core = rng.integers(0, 4, int(length), dtype=np.uint8)
        k = int(rng.integers(22, 40))
        at = int(rng.integers(0, max(1, int(length) - k)))
        left, seed, right = core[:at], core[at:at + k], core[at + k:]
        other = [_mutate(rng, left, case["rate"]), seed, _mutate(rng, right, case["rate"])]
        hang = [rng.integers(0, 4, int(rng.integers(0, length // 2 + 1)), dtype=np.uint8) for _ in range(2)]
        s, t = [left, seed, right], other
        start, offset = len(left), len(other[0])
        s.append(hang[0]) if rng.random() < 0.5 else t.append(hang[0])
        if rng.random() < 0.5:
            s.insert(0, hang[1])
            start += len(hang[1])
        else:
            t.insert(0, hang[1])
            offset += len(hang[1])
        s, t = np.concatenate(s), np.concatenate(t)
        s_dir = int(rng.integers(0, 2))
        seqs += [3 - s[::-1] if s_dir else s, t]
        tasks.append((len(seqs) - 1, len(seqs), s_dir, start, offset, k))
    return seqs, np.array(tasks, oic.EXT_TASK)


def _prepare_dp(case, rng):
    bound, limits = oic.dp_tables(case["maxerate"])
    seqs, tasks = [], []
    for i, length in enumerate(_lengths(rng, case["tasks"], case["length"])):
        a = rng.integers(0, 4, int(length), dtype=np.uint8)
        b = _mutate(rng, a, case["rate"])
        if rng.random() < 0.3:
            b = np.concatenate([b, rng.integers(0, 4, int(rng.integers(0, 200)), dtype=np.uint8)])
        seqs += [a, b]
        ia, ib = (2 * i + 1, 2 * i + 2) if len(a) <= len(b) else (2 * i + 2, 2 * i + 1)
        m, n = min(len(a), len(b)), max(len(a), len(b))
        limit = min(int(bound[m]) + 3, len(limits) - 1, 1021)
        back = i % 2
        tasks.append((ia, ib, 0, 0, (m - 1) * back, (n - 1) * back, m, n, limit, back))
    return seqs, np.array(tasks, oic.DP_TASK)


def _traces(case, rng):
    """Features of candidate pairs (mixed scales) and a smooth cost of them with noise; the last tenth is held out."""
    n = case["samples"] + case["samples"] // 9
    feat = rng.normal(0.0, 1.0, (n, oic.NFEAT)).astype(np.float32) * np.linspace(0.3, 3.0, oic.NFEAT, dtype=np.float32) + 2.0
    mix = rng.normal(0.0, 0.4, (oic.NFEAT, oic.NOUT)).astype(np.float32)
    targ = (np.tanh(feat @ mix) * 3.0 + rng.normal(0.0, 0.1, (n, oic.NOUT))).astype(np.float32)
    return feat, targ


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "train":
        feat, targ = _traces(case, rng)
        cut = case["samples"]
        return dict(kind=kind, eng=oic.Engine(maxerate=0.045), train=(feat[:cut], targ[:cut]), test=feat[cut:], batch=case["batch"],
                    epochs=case["epochs"])
    if kind in ("job", "search"):
        reads = readsim.simulate(readsim.PRESETS[case["preset"]].scaled(case["genome"], seed=1 + seed))
        eng = oic.Engine(schedule=SCHEDULES[case["schedule"]], threads=1, partial=bool(case.get("partial")), **OPTIONS[case["preset"]])
        out = np.zeros((MAX_RECORDS, 3), np.int64)
        if kind == "job":
            return dict(kind=kind, eng=eng, reads=reads, last_ref=case["last_ref"] or reads.n, out=out, filled=0)
        eng.load_reads(reads)
        eng.build_hash_index(1, reads.n)
        return dict(kind=kind, eng=eng, last_ref=min(case["refs"], reads.n), counters=eng.counters(), out=out, filled=0)
    seqs, tasks = _prepare_extend(case, rng) if kind == "extend" else _prepare_dp(case, rng)
    reads = _read_set(seqs)
    eng = oic.Engine(maxerate=case["maxerate"], minlength=40)
    eng.load_reads(reads)
    # a task's delta is no longer than its error limit; a read (with its hangs) is at most 8 mean lengths
    stride = 64 + int(math.ceil(8 * case["length"] * case["maxerate"]))
    stride = min(stride, 1024 if kind != "extend" else 4096, (1 << 20) // len(tasks))
    return dict(kind=kind, eng=eng, tasks=tasks, stride=stride, res=np.zeros(len(tasks), oic.DP_RESULT),
                delta=np.zeros((len(tasks), stride), np.int32), out=np.zeros(len(tasks) * stride, np.int32), filled=0)


COUNTED = ("hits", "pairs", "nodes", "extensions", "dp_cells")


def run(state):
    kind, eng = state["kind"], state["eng"]
    if kind == "train":
        feat, targ = state["train"]
        loss = eng.train_model(feat, targ, epochs=state["epochs"], batch=state["batch"])
        weights, mu, sd = eng.model()
        return dict(loss=loss, weights=weights, mu=mu, sd=sd, predicted=eng.predict(state["test"]))
    if kind == "job":
        eng.load_reads(state["reads"])
        r = eng.run(1, 0xFFFFFFFF, 1, state["last_ref"])
        return dict(records=_keep(state, _plain(r.records)), stats=np.array(r.stats, np.int64), counted=np.array([r.counters[k] for k in COUNTED], np.int64))
    if kind == "search":
        before = state["counters"]
        r = eng.search(1, state["last_ref"])
        state["counters"] = r.counters            # they run on from search to search
        return dict(records=_keep(state, _plain(r.records)), stats=np.array(r.stats, np.int64),
                    counted=np.array([r.counters[k] - before[k] for k in COUNTED], np.int64))
    if kind == "extend":
        res, delta = eng.extend_alignment(state["tasks"], delta_stride=state["stride"])
    elif kind == "dp":
        res, delta = eng.prefix_dp(state["tasks"], delta_stride=state["stride"])
    else:
        res, delta, tasks = state["res"], state["delta"], state["tasks"]
        rc = oic.lib().oic_prefix_dp_batch_noalloc(eng._ctx, tasks.ctypes.data, len(tasks), res.ctypes.data, delta.ctypes.data,
                                                   ctypes.c_uint32(state["stride"]))
        if rc != oic.OIC_OK:
            raise oic.OicError(rc, oic.lib().oic_last_error(eng._ctx).decode())
        res = res.copy()
    # each task's delta has delta_len entries and nothing is defined past them: packed one after another
    used = np.concatenate([d[:n] for d, n in zip(delta, res["delta_len"])])
    return dict(results=res.view(np.int32).reshape(len(res), -1), deltas=_keep(state, used))


def _keep(state, rows):
    """The rows in the state's own output buffer, zeros after them."""
    out, last = state["out"], state["filled"]
    n = state["filled"] = len(rows)
    out[:n] = rows
    out[n:last] = 0
    return out


def _plain(records):
    """24-byte records as rows of three 64-bit words."""
    return records.view(np.int64).reshape(-1, 3)


def work(case):
    """Bytes: inputs in, outputs out, and a job's table and a search's ref reads once.  Operations: 4 per DP cell
    (the recurrence) and 2 per 16 bases compared, or the model's products."""
    kind = case["kind"]
    if kind == "train":
        per = 2 * (12 * 64 + 64 * 64 + 64 * 2)
        n = case["samples"]
        return dict(bytes=float(n * 56 * (case["epochs"] + 1)), flops=float(per * (3 * n * case["epochs"] + n // 9)))
    if kind in ("job", "search"):
        cfg = readsim.PRESETS[case["preset"]]
        mean = math.exp(cfg.ln_mu + cfg.ln_sigma ** 2 / 2) * (0.75 if cfg.hpc else 1.0)
        total = case["genome"] * cfg.coverage * (0.75 if cfg.hpc else 1.0)
        refs = case.get("refs") or case["last_ref"]
        ref_bases = min(total, refs * mean) if refs else total / 2      # a pair is found from its lower read
        ops = 4.0 * CELLS[case["preset"]] * ref_bases
        # both strands packed (1/2 B), 8 B per indexed position
        return dict(bytes=(total * 9.5 if kind == "job" else 0.0) + 16.0 * ref_bases, flops=ops)
    # both tails' rows up to the errors at hand, bands about twice as wide as the drift of the errors
    errors = case["length"] * min(case["rate"], case["maxerate"])
    cells = case["tasks"] * errors * min(2.0 * errors + 1.0, 40.0)
    return dict(bytes=case["tasks"] * (2.0 * case["length"] / 4 + 4 * errors + 40), flops=4.0 * cells)


def exact(case, seed):
    """The standardisation in 64 bits.  Everything else that is not a whole number follows from weights that the
    library draws and from samples that it shuffles by its own seeded generator."""
    if case["kind"] != "train":
        return None
    feat = _traces(case, np.random.default_rng(seed))[0][:case["samples"]].astype(np.float64)
    return dict(loss=None, weights=None, mu=feat.mean(axis=0), sd=feat.std(axis=0), predicted=None)
