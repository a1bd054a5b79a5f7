"""Small calls at the edges of their inputs."""
import ctypes

import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

TOL = 1e-3  # the parity bar; rows x columns as in test_gpu_small


def _seq(rng, n, letters="ACGT"):
    return "".join(rng.choice(list(letters), n))


NAMES = ("read_data", "hap_data", "base_quals", "ins_quals", "del_quals", "gcp_quals",
         "read_lengths", "hap_lengths", "read_offsets", "hap_offsets", "num_reads_per_group",
         "num_haps_per_group", "reads_prefix", "haps_prefix")


def _batch(rng, records):
    """A batch of (reads, haps) records, sequences given as text, which may be
    empty; qualities 2 to 40, gaps 45 or, every other read, 25 to 45."""
    import gpupairhmm_amd as G
    reads = [r for rs, _ in records for r in rs]
    haps = [h for _, hs in records for h in hs]

    def pack(seqs, make, pad):
        out = []
        for i, s in enumerate(seqs):
            out.append(np.asarray(make(i, s), np.uint8))
            out.append(np.full(4 - len(s) % 4, pad, np.uint8))
        return np.concatenate(out)

    def offsets(seqs):
        return np.concatenate([[0], np.cumsum([len(s) + 4 - len(s) % 4 for s in seqs])])

    def text(_, s):
        return np.frombuffer(s.encode(), np.uint8)

    def gaps(i, s):
        return np.full(len(s), 45) if i % 2 == 0 else rng.integers(25, 46, len(s))

    gap = pack(reads, gaps, 45)
    return G.HostBatch.from_arrays(
        read_data=pack(reads, text, ord("N")), hap_data=pack(haps, text, ord("N")),
        base_quals=pack(reads, lambda i, s: rng.integers(2, 41, len(s)), 45),
        ins_quals=gap, del_quals=gap,
        gcp_quals=pack(reads, lambda i, s: np.full(len(s), 10), 45),
        read_lengths=[len(r) for r in reads], hap_lengths=[len(h) for h in haps],
        read_offsets=offsets(reads), hap_offsets=offsets(haps),
        num_reads_per_group=[len(rs) for rs, _ in records],
        num_haps_per_group=[len(hs) for _, hs in records],
        reads_prefix=np.concatenate([[0], np.cumsum([len(rs) for rs, _ in records])]),
        haps_prefix=np.concatenate([[0], np.cumsum([len(hs) for _, hs in records])]))


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("semantics", [0, 1])
def test_empty_reads_and_haps(lib, oracle, semantics):
    """Empty reads, the batch's first among them (whose packed row nothing
    writes, and lanes without a read load it), empty haps and records of
    nothing else: -inf where the oracle says so, on every route."""
    import gpupairhmm_amd as G
    rng = np.random.default_rng(41)
    hap = _seq(rng, 260)
    b = _batch(rng, [
        (["", hap[:150], "", hap[40:190]], [hap, "", _seq(rng, 90), ""]),
        (["", ""], [hap[:70], ""]),
        ([hap[:30]], [""]),
        ([hap[10:110], "", hap[:61]] + [hap[i:i + 101] for i in range(20)], ["", hap, hap[:200] + "N"]),
        (["", _seq(rng, 1100)], [_seq(rng, 1200), ""]),
    ])
    say(f"case: empty reads and haps, semantics {semantics}, {b.num_alignments} alignments")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=semantics)
    fin = np.isfinite(ref)
    assert 0 < fin.sum() < len(ref)
    with G.Engine(semantics=semantics, mode=G.MODE_PLAIN) as e:
        want = e.score_batch(b)
    assert np.all(want[~fin] == -np.inf)
    assert np.max(np.abs(want[fin].astype(np.float64) - ref[fin])) <= TOL
    for kw in ({}, {"graphs": False}, {"small_batch": 0}, {"time_kernels": True}):
        with G.Engine(semantics=semantics, **kw) as e:
            got = e.score_batch(b)
            assert np.all(got[~fin] == -np.inf)
            assert np.max(np.abs(got[fin].astype(np.float64) - ref[fin])) <= TOL
            if "small_batch" not in kw:
                assert np.array_equal(_bits(got), _bits(want)), kw
            db, out = e.upload(b), e.alloc(4 * b.num_alignments)
            e.score_device_noalloc(db, out)
            e.synchronize()
            assert np.array_equal(_bits(e.download(out, b.num_alignments)), _bits(got)), kw
            e.free(out)
            db.free()


def test_server_launches_fit_the_reservation(lib):
    """A server's launch contexts are reserved at creation for the largest
    launch; merged launches of every size below it, among them small calls on
    either side of the powers of two of their lists' capacity, take no more
    device memory and capture no graph anew."""
    import gpupairhmm_amd as G

    def free_bytes():  # the library's own HIP runtime
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    rng = np.random.default_rng(43)
    reads = [_seq(rng, 40) for _ in range(500)]
    sizes = (40000, 65500, 66000, 131000, 131500, 262000)
    batches = [_batch(rng, [(reads, [_seq(rng, 60) for _ in range(n // 500)])]) for n in sizes]
    with G.Engine() as e:
        alone = [e.score_batch(b) for b in batches]
    with G.Engine() as e:
        srv = G.Server(e, hbm_budget_bytes=4 << 30)
        try:
            seen = []
            for n, b, want in zip(sizes, batches, alone):
                say(f"case: server launch of {n} alignments")
                assert srv.submit(b, n)
                tag, got, _ = srv.poll(timeout_ms=20000, capacity=n)
                assert tag == n and np.array_equal(_bits(got), _bits(want))
                seen.append((free_bytes(), e.stats().graph_captures))
            assert len(set(seen)) == 1, seen
        finally:
            srv.close()


def _steep(rng, lens):
    """Reads hanging over their haps under a gap continuation of 40, which the
    in-pass scaling mostly refuses; the last one lies within its hap."""
    recs = []
    for L in lens:
        ref = _seq(rng, L + 200)
        recs.append(([ref[o:o + L] for o in (0, 30, 60, 200)],
                     [ref[90:], ref[:max(8, L // 2)], ref[L // 3:L + 100], ref]))
    b = _batch(rng, recs)
    b.gcp_quals[:] = 40
    return b


@pytest.mark.parametrize("f64_rows", [0, 4, 6, 8, 10])
@pytest.mark.parametrize("lens", [(20, 79, 80, 150, 511), (512, 600, 1023)])
def test_fp64_of_small_calls(lib, oracle, lens, f64_rows):
    """What the in-pass scaling refuses is recomputed in FP64: reads of up to
    511 bases in tiles, of f64_rows rows per lane where the option names them,
    the others on waves."""
    import gpupairhmm_amd as G
    b = _steep(np.random.default_rng(47), lens)
    say(f"case: FP64 of small calls, reads of {lens}, f64_rows {f64_rows}")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=1)
    assert np.all(np.isfinite(ref))
    want = None
    for kw in ({}, {"graphs": False}):
        with G.Engine(semantics=1, f64_rows=f64_rows, **kw) as e:
            got = e.score_batch(b)
            st = e.stats()
        assert st.f64_alignments >= len(ref) // 4
        want = got if want is None else want
        assert np.array_equal(_bits(got), _bits(want))
    # the parity bar, and a float's own step for scores in the thousands
    assert np.all(np.abs(got.astype(np.float64) - ref) <= TOL + np.spacing(np.abs(ref).astype(np.float32)))


# hap columns per wave at 256 compute units, as the few-launch sequence of small
# calls reckons them: on either side of its limits for records of few reads and
# of many, and of the number at which its hap segments shrink
@pytest.mark.parametrize("reads,haps,hap_len,columns", [
    (25, 4, 250, (1560, 1640)), (64, 30, 300, (1900, 2200)), (64, 30, 300, (4050, 4140))])
def test_column_limits(lib, reads, haps, hap_len, columns):
    import gpupairhmm_amd as G
    rng = np.random.default_rng(53)
    hap = [_seq(rng, hap_len) for _ in range(haps)]
    read = [hap[0][o:o + 147] for o in rng.integers(0, hap_len - 147, reads)]
    per_record = reads * haps * (hap_len + 4 - hap_len % 4) / 6 / 2048  # six reads side by side
    counts = [int(c / per_record) + 1 for c in columns]
    for n in counts:
        b = _batch(rng, [(read, hap)] * n)
        say(f"case: {n} records of {reads} x {haps}, {n * per_record:.0f} columns per wave")
        with G.Engine(mode=G.MODE_PLAIN) as e:
            want = e.score_batch(b)
        with G.Engine() as e:
            got = e.score_batch(b)
        assert np.all(np.isfinite(want)) and np.array_equal(_bits(got), _bits(want))
