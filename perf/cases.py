"""The work that users of this framework have it do, as cases to be timed.

A case describes one call (or one burst of requests): how many records, how
many reads and haplotypes each holds, their lengths and qualities, the entry
point and the gap semantics.  ``prepare`` makes the inputs from a seed and puts
them where such a program holds them, ``run`` makes one pass, ``exact`` gives
the same scores in 64 bits.  Engines and servers are made once per process and
kept, as a program keeps them; inputs are new for every ``prepare``.

Inputs follow the model of the package's synthetic workloads: a record has a
random reference, haplotypes are mutated copies of it, reads are drawn from the
haplotypes with substitution errors.
"""
import functools
import math

import numpy as np
import torch

import gpupairhmm_amd as G

_BASES = np.frombuffer(b"ACGT", dtype=np.uint8)
_SEMANTICS = {"gpu": G.SEM_GPU, "cpu": G.SEM_CPU, "gcp": G.SEM_GCP}

# What a case is unless it says otherwise: device-resident scoring of records
# of the mixed-length workload's kind.
_DEFAULTS = {
    "entry": "device",       # device | host | region | serve
    "semantics": "gpu",      # gpu | cpu | gcp
    "records": 1,
    "reads_min": 1, "reads_max": 500,
    "haps_min": 1, "haps_max": 64,
    "read_median": 150, "read_sigma": 0.35, "read_min": 36, "read_max": 300,
    "hap_extra": 100,        # > 0: record's median read length + lognormal(hap_extra, 0.5)
    "hap_min": 1, "hap_max": 1000,
    "q_min": 10, "q_max": 40, "errors": 0.01,
    "indel_quals": "flat",   # flat: 40, the last 45; varying: a quality of its own per base
    "gcp": "flat",           # flat: 10; varying: a gap continuation of its own per base
    "n_haps": 0.0,           # share of haplotypes that hold a run of N
}


def _full(case):
    return {**_DEFAULTS, **case}


def _fixed(reads, haps, read_len, hap_min, hap_max):
    return {"reads_min": reads, "reads_max": reads, "haps_min": haps, "haps_max": haps,
            "read_sigma": 0.0, "read_min": read_len, "read_max": read_len, "hap_extra": 0,
            "hap_min": hap_min, "hap_max": hap_max}


def listed():
    return [
        # one small active region from an in-process variant caller (its own
        # gap-continuation semantics): the smallest call, all latency
        {"name": "region_call", "entry": "region", "semantics": "cpu",
         **_fixed(8, 4, 100, 120, 120)},
        # one ordinary region, resident on the device
        {"name": "one_region", "reads_min": 250, "reads_max": 250, "haps_min": 32, "haps_max": 32},
        # many small regions in one call (the CPU-runnable workload)
        {"name": "short_batch", "records": 1000, **_fixed(8, 4, 100, 120, 120)},
        # a sequencer's fixed 150-base reads, a million alignments, device-resident ...
        {"name": "fixed_150", "records": 10000, **_fixed(25, 4, 150, 150, 350)},
        # ... and the same from the caller's host arrays to host scores
        {"name": "fixed_150_host", "records": 10000, "entry": "host",
         **_fixed(25, 4, 150, 150, 350)},
        # the headline workload's records: everything mixed, a large batch
        {"name": "mixed", "records": 1000},
        # low-quality long-window work: 250-base reads against haps of 2-5 kb
        {"name": "long_haps", "records": 400, "q_min": 2, "q_max": 20, "errors": 0.05,
         **_fixed(16, 8, 250, 2000, 5000)},
        # recalibrated reads: insertion and deletion qualities that differ from base to base
        {"name": "indel_quals", "records": 100, "indel_quals": "varying"},
        # every position with its own gap continuation
        {"name": "gcp_per_base", "records": 100, "semantics": "gcp", "gcp": "varying"},
        # reads longer than the largest tile (the multi-tile path)
        {"name": "long_reads", "records": 40, **_fixed(16, 4, 1300, 1500, 2000),
         "read_min": 1100, "read_max": 1500},
        # windows whose reference holds Ns: some haplotypes carry the wildcard
        {"name": "wildcard_haps", "records": 100, "n_haps": 0.05},
        # a burst of independent region requests to the serving loop
        {"name": "serve_burst", "records": 128, "entry": "serve"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("region", "one", "short", "fixed", "fixed", "host", "mixed", "mixed",
                       "long_haps", "indel", "gcp", "cpu", "long_reads", "wildcard", "serve"))
    if kind == "region":
        return {"entry": "region", "semantics": rng.choice(("cpu", "gpu")),
                **_fixed(rng.randint(1, 64), rng.randint(1, 16), rng.randint(36, 300),
                         rng.randint(40, 200), rng.randint(200, 500))}
    if kind == "one":
        r, h = _log_int(rng, 20, 500), rng.randint(2, 64)
        return {"reads_min": r, "reads_max": r, "haps_min": h, "haps_max": h}
    if kind == "short":
        return {"records": _log_int(rng, 50, 4000),
                **_fixed(rng.randint(3, 20), rng.randint(2, 8), rng.randint(50, 151),
                         rng.randint(100, 150), rng.randint(150, 250))}
    if kind in ("fixed", "host"):
        return {"records": _log_int(rng, 300, 10000), "entry": "host" if kind == "host" else "device",
                **_fixed(rng.randint(10, 40), rng.randint(2, 6), rng.choice((76, 100, 101, 125, 150, 151, 250)),
                         rng.randint(150, 250), rng.randint(260, 400))}
    if kind == "long_haps":
        return {"records": _log_int(rng, 20, 1000), "q_min": 2, "q_max": rng.randint(20, 40),
                "errors": round(rng.uniform(0.01, 0.05), 3),
                **_fixed(rng.randint(8, 24), rng.randint(4, 10), rng.randint(150, 300),
                         rng.randint(1000, 2000), rng.randint(2000, 5000))}
    if kind == "long_reads":
        lo = rng.randint(1050, 1400)
        return {"records": _log_int(rng, 4, 60),
                **_fixed(rng.randint(4, 20), rng.randint(2, 5), lo, lo + 100, lo + rng.randint(200, 900)),
                "read_max": lo + rng.randint(50, 500)}
    if kind == "serve":
        return {"records": _log_int(rng, 8, 200), "entry": "serve"}
    case = {"records": _log_int(rng, 10, 800 if kind == "mixed" else 200),
            "read_median": rng.randint(90, 220)}
    if kind == "indel":
        case["indel_quals"] = "varying"
    elif kind == "gcp":
        case.update(semantics="gcp", gcp="varying")
    elif kind == "cpu":
        case["semantics"] = "cpu"
    elif kind == "wildcard":
        case["n_haps"] = round(rng.uniform(0.01, 0.1), 3)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _prefix(x):
    return np.concatenate([[0], np.cumsum(x, dtype=np.int64)])


def _within(lens):
    """0 .. len-1 for each of `lens`, one after another."""
    total = int(lens.sum())
    return np.arange(total, dtype=np.int64) - np.repeat(_prefix(lens)[:-1], lens)


def _shape(case, rng):
    """Records' read and hap counts (the case's own, so that its scores have one
    shape whatever the seed), and every read's and hap's length."""
    n = case["records"]
    counts = np.random.default_rng(n)
    R = counts.integers(case["reads_min"], case["reads_max"] + 1, n)
    H = counts.integers(case["haps_min"], case["haps_max"] + 1, n)
    nr, nh = int(R.sum()), int(H.sum())
    if case["read_sigma"] > 0:
        rl = np.rint(case["read_median"] * np.exp(case["read_sigma"] * rng.standard_normal(nr)))
        rl = np.clip(rl, case["read_min"], case["read_max"]).astype(np.int64)
    else:
        rl = rng.integers(case["read_min"], case["read_max"] + 1, nr)
    if case["hap_extra"] > 0:
        rec = np.repeat(np.arange(n), R)
        median = rl[np.lexsort((rl, rec))][_prefix(R)[:-1] + R // 2]
        extra = np.rint(case["hap_extra"] * np.exp(0.5 * rng.standard_normal(nh)))
        hl = np.clip(np.repeat(median, H) + extra, case["hap_min"], case["hap_max"]).astype(np.int64)
    else:
        hl = rng.integers(case["hap_min"], case["hap_max"] + 1, nh)
    return R, H, rl, hl


def _arrays(case, seed):
    """The batch's arrays in the framework's layout (padded sequences, qualities
    less 33), named as HostBatch.from_arrays names them."""
    rng = np.random.default_rng(int(seed))
    R, H, rl, hl = _shape(case, rng)
    n, rp, hp = len(R), _prefix(R), _prefix(H)
    # each record's reference
    ref_len = np.maximum(np.maximum.reduceat(hl, hp[:-1]), np.maximum.reduceat(rl, rp[:-1])) + 64
    ref_at = _prefix(ref_len)
    ref = rng.integers(0, 4, int(ref_at[-1]), dtype=np.uint8)
    # haplotypes: a walk over the reference with 0.1% insertions (a stretch
    # repeated) and 0.1% deletions of 1-5 bases, and 1% substitutions
    hap_at = _prefix(hl)
    nb = int(hap_at[-1])
    step = np.ones(nb, dtype=np.int64)
    for sign in (-1, 1):
        at = rng.integers(0, nb, rng.binomial(nb, 0.001))
        step[at] = 1 + sign * rng.integers(1, 6, len(at))
    walk = np.cumsum(step)
    walk -= np.repeat(walk[hap_at[:-1]], hl)
    rec_h = np.repeat(np.arange(n), H)
    walk = np.clip(walk, 0, np.repeat(ref_len[rec_h] - 1, hl)) + np.repeat(ref_at[rec_h], hl)
    haps = ref[walk]
    at = rng.integers(0, nb, rng.binomial(nb, 0.01))
    haps[at] = (haps[at] + rng.integers(1, 4, len(at), dtype=np.uint8)) & 3
    # reads: from a random haplotype of the record at a random offset (from
    # the reference where that haplotype is too short)
    rec_r = np.repeat(np.arange(n), R)
    src = hp[rec_r] + rng.integers(0, H[rec_r])
    room = hl[src] - rl
    u = rng.random(len(rl))
    start = np.where(room >= 0, hap_at[src] + (u * (room + 1)).astype(np.int64),
                     nb + ref_at[rec_r] + (u * (ref_len[rec_r] - rl + 1)).astype(np.int64))
    reads = np.concatenate([haps, ref])[np.repeat(start, rl) + _within(rl)]
    nrb = len(reads)
    at = rng.integers(0, nrb, rng.binomial(nrb, case["errors"]))
    reads[at] = (reads[at] + rng.integers(1, 4, len(at), dtype=np.uint8)) & 3
    # the padded layout: len + (4 - len % 4) bytes, padding 'N' and quality 45
    rpad, hpad = rl + 4 - rl % 4, hl + 4 - hl % 4
    ro, ho = _prefix(rpad), _prefix(hpad)
    rslot = np.repeat(ro[:-1], rl) + _within(rl)
    hslot = np.repeat(ho[:-1], hl) + _within(hl)

    def quals(values):
        out = np.full(int(ro[-1]), 45, dtype=np.uint8)
        out[rslot] = values
        return out

    def indel():
        if case["indel_quals"] == "varying":
            return quals(rng.integers(30, 46, nrb, dtype=np.uint8))
        q = np.full(nrb, 40, dtype=np.uint8)
        q[_prefix(rl)[1:] - 1] = 45
        return quals(q)

    read_data = np.full(int(ro[-1]), ord("N"), dtype=np.uint8)
    read_data[rslot] = _BASES[reads]
    hap_data = np.full(int(ho[-1]), ord("N"), dtype=np.uint8)
    hap_data[hslot] = _BASES[haps]
    for k in np.flatnonzero(rng.random(len(hl)) < case["n_haps"]):
        at = int(ho[k]) + int(rng.integers(0, hl[k]))
        hap_data[at:min(at + int(rng.integers(1, 6)), int(ho[k] + hl[k]))] = ord("N")
    return {
        "read_data": read_data, "hap_data": hap_data,
        "base_quals": quals(rng.integers(case["q_min"], case["q_max"] + 1, nrb, dtype=np.uint8)),
        "ins_quals": indel(), "del_quals": indel(),
        "gcp_quals": quals(rng.integers(8, 21, nrb, dtype=np.uint8)
                           if case["gcp"] == "varying" else np.uint8(10)),
        "read_lengths": rl.astype(np.int32), "hap_lengths": hl.astype(np.int32),
        "read_offsets": ro.astype(np.int32), "hap_offsets": ho.astype(np.int32),
        "num_reads_per_group": R.astype(np.int32), "num_haps_per_group": H.astype(np.int32),
        "reads_prefix": rp.astype(np.int32), "haps_prefix": hp.astype(np.int32)}


# ---------------------------------------------------------------------------
# the framework
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _engine(semantics):
    return G.Engine(mode=G.MODE_BATCHED, semantics=_SEMANTICS[semantics])


@functools.lru_cache(maxsize=None)
def _server(semantics):
    return G.Server(_engine(semantics), hbm_budget_bytes=8 << 30)


def prepare(case, seed):
    case = _full(case)
    eng = _engine(case["semantics"])
    a = _arrays(case, seed)
    batch = G.HostBatch.from_arrays(**a)
    state = {"entry": case["entry"], "engine": eng, "batch": batch}
    if case["entry"] == "device":
        # inputs and scores stay on the device, on the engine's own stream
        state["resident"] = eng.upload(batch)
        state["scores"] = torch.empty(batch.num_alignments, dtype=torch.float32, device="cuda")
    elif case["entry"] == "region":
        # a caller's own objects: one tuple of arrays per read, one array per hap
        quals = ("read_data", "base_quals", "ins_quals", "del_quals", "gcp_quals")
        state["reads"] = [tuple(a[k][o:o + n].copy() for k in quals)
                          for o, n in zip(a["read_offsets"], a["read_lengths"])]
        state["haps"] = [a["hap_data"][o:o + n].copy()
                         for o, n in zip(a["hap_offsets"], a["hap_lengths"])]
    elif case["entry"] == "serve":
        state["server"] = _server(case["semantics"])
        state["requests"] = [batch.subset([g]) for g in range(batch.num_groups)]
    return state


def run(state):
    entry, eng = state["entry"], state["engine"]
    if entry == "device":
        eng.score_device(state["resident"], state["scores"].data_ptr())
        return state["scores"]
    if entry == "host":
        return eng.score_batch(state["batch"])
    if entry == "region":
        # FP32 scores, which this entry point hands out widened
        return eng.compute_likelihoods(state["reads"], state["haps"]).astype(np.float32).reshape(-1)
    server, requests = state["server"], state["requests"]
    scores = [None] * len(requests)
    for tag, request in enumerate(requests):
        if not server.submit(request, tag):
            raise RuntimeError("the server refused a request of a burst that fits its budget")
    for _ in requests:
        tag, got, _ = server.poll(timeout_ms=20000)
        scores[tag] = got
    return np.concatenate(scores)


def _lengths(case):
    R, H, rl, hl = _shape(case, np.random.default_rng(0))
    rp, hp = _prefix(R), _prefix(H)
    cells = int((np.add.reduceat(rl, rp[:-1]) * np.add.reduceat(hl, hp[:-1])).sum())
    return R, H, rl, hl, cells


def work(case):
    """Each base and quality read once and each score written once; 11
    operations per cell of the recurrence (M 5, I 3, D 3)."""
    case = _full(case)
    R, H, rl, hl, cells = _lengths(case)
    per_base = 5 if case["semantics"] != "gpu" else 4
    return {"bytes": int(per_base * rl.sum() + hl.sum() + 4 * (R * H).sum()), "flops": 11 * cells}


# ---------------------------------------------------------------------------
# the same scores in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    """log10 of the forward sum for every (read, hap) pair, read-major within a
    record: the recurrence in float64 logarithms, one anti-diagonal of many
    alignments at a time."""
    case = _full(case)
    if _lengths(case)[4] > 5e10:
        return None
    a = _arrays(case, seed)
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    R, H = a["num_reads_per_group"].astype(np.int64), a["num_haps_per_group"].astype(np.int64)
    rp, hp = _prefix(R), _prefix(H)
    per = R * H
    rec = np.repeat(np.arange(len(R)), per)
    k = _within(per)
    read = torch.from_numpy(rp[rec] + k // H[rec]).to(dev)
    hap = torch.from_numpy(hp[rec] + k % H[rec]).to(dev)
    t = {name: torch.from_numpy(v).to(dev) for name, v in a.items()}
    rl, hl = t["read_lengths"].long(), t["hap_lengths"].long()
    order = torch.argsort(rl[read] * 65536 + hl[hap])
    out = torch.empty(len(rec), dtype=torch.float64, device=dev)
    at = 0
    while at < len(rec):
        # a chunk of alignments of similar lengths
        count = min(len(rec) - at, max(1, 20_000_000 // int(rl[read[order[-1]]] + 1)))
        ids = order[at:at + count]
        out[ids] = _forward(case, t, read[ids], hap[ids], rl, hl)
        at += count
    return out.to("cpu") if case["entry"] != "device" else out


def _forward(case, t, read, hap, rl, hl):
    dev, neg = read.device, -math.inf
    L, HL = rl[read], hl[hap]
    B, Lmax, Hmax = len(read), int(L.max()), int(HL.max())
    row = torch.arange(Lmax, device=dev)
    inside = row[None, :] < L[:, None]
    base = torch.where(inside, t["read_offsets"][read].long()[:, None] + row, 0)

    def p(name):
        return torch.pow(10.0, -t[name][base].double() / 10.0)

    err, ins, dele = p("base_quals"), p("ins_quals"), p("del_quals")
    if case["semantics"] == "gpu":
        eps = torch.full((B, 1), 0.1, dtype=torch.float64, device=dev)
    elif case["semantics"] == "cpu":
        eps = p("gcp_quals")[:, :1]
    else:
        eps = p("gcp_quals")
    log_eps, log_beta = eps.log(), (1 - eps).log()
    log_alpha, log_ins, log_del = (1 - (ins + dele)).log(), ins.log(), dele.log()
    hit, miss = (1 - err).log(), (err / 3).log()
    bases = t["read_data"][base]
    miss = torch.where(bases == ord("N"), hit, miss)
    # haps right to left, so that an anti-diagonal reads them in row order:
    # row r (0-based) of diagonal d meets column d - 2 - r (0-based), which is
    # entry Hmax - 1 - (d - 2 - r) of the reversed hap
    col = torch.arange(Hmax - 1, -1, -1, device=dev)
    ok = col[None, :] < HL[:, None]
    letters = t["hap_data"][torch.where(ok, t["hap_offsets"][hap].long()[:, None] + col, 0)]
    letters = torch.where(ok, letters, ord("N"))
    pad = torch.full((B, Lmax), ord("N"), dtype=letters.dtype, device=dev)
    letters = torch.cat([pad, letters, pad], 1)
    start = -HL.double().log()
    # M, I, D of the last two diagonals, row 0 first
    M, I, D = ([torch.full((B, Lmax + 1), neg, dtype=torch.float64, device=dev) for _ in range(3)]
               for _ in range(3))
    for x in D:
        x[:, 0] = start
    total = torch.full((B,), neg, dtype=torch.float64, device=dev)
    last = L[:, None]
    for d in range(2, Lmax + Hmax + 1):
        n, o, oo = d % 3, (d - 1) % 3, (d - 2) % 3  # this diagonal and the two before
        lo, hi = max(1, d - Hmax), min(Lmax, d - 1)  # rows with a column in 1 .. Hmax
        up, at, k = slice(lo - 1, hi), slice(lo, hi + 1), slice(lo - 1, hi)
        first = Lmax + Hmax - 1 - (d - 2) + (lo - 1)
        h = letters[:, first:first + hi - lo + 1]
        lam = torch.where((h == bases[:, k]) | (h == ord("N")), hit[:, k], miss[:, k])
        e = log_eps if log_eps.shape[1] == 1 else log_eps[:, k]
        b = log_beta if log_beta.shape[1] == 1 else log_beta[:, k]
        M[n][:, at] = lam + torch.logaddexp(log_alpha[:, k] + M[oo][:, up],
                                            b + torch.logaddexp(I[oo][:, up], D[oo][:, up]))
        I[n][:, at] = torch.logaddexp(log_ins[:, k] + M[o][:, up], e + I[o][:, up])
        D[n][:, at] = torch.logaddexp(log_del[:, k] + M[o][:, at], e + D[o][:, at])
        end = torch.logaddexp(M[n].gather(1, last), I[n].gather(1, last))[:, 0]
        c = d - L
        total = torch.where((c >= 1) & (c <= HL), torch.logaddexp(total, end), total)
    return total / math.log(10.0)
