"""Scores of reads of several tiles against the FP64 oracle, to the precision of
a float rather than to the parity bar: what falls below the FP32 range was an
FP64 recompute before the strips took it, and has to be as good.

Tolerance, log10.  Along its best path a score takes five FP32 roundings a row,
each within 2^-24 of the value and as often up as down: a standard deviation of
0.4343 * sqrt(5 L) * 2^-24 / sqrt(3) = 1.6e-6 at 2,304 rows, five of which are
allowed (8e-6), beside half a unit of the float that holds the score.  What adds
up over the rows instead -- every row of equal qualities rounds its factors the
same way, here up to 2.6e-5 over 1,500 rows -- may leave 3e-6, for the rows in
which a path is not in a match; the mean over many scores, where the rest
cancels, is held to that."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

DRIFT, PATH = 3e-6, 8e-6
LOW = -75.3  # FP32 sums below FLT_MIN


def _seq(rng, n):
    return "".join(rng.choice(list("ACGT"), n))


def _noisy(rng, s, err):
    s = list(s)
    for i in np.flatnonzero(rng.random(len(s)) < err):
        s[i] = "ACGT"[int(rng.integers(4))]
    return "".join(s)


def _phred(q):
    return "".join(chr(33 + int(x)) for x in q)


@pytest.mark.parametrize("semantics", [0, 1])
@pytest.mark.parametrize("ins", [(40, 40), (44, 27)])  # the second: no rescaled form
def test_precision(lib, oracle, semantics, ins):
    import gpupairhmm_amd as G
    rng = np.random.default_rng(61)
    text = ""
    for L in (1024, 1100, 1400, 1535, 1536, 2304):
        lines, ref = [], _seq(rng, L + 150)
        for o in range(0, 150, 15):
            iq = np.where(np.arange(L) % 2 == 0, ins[0], ins[1])
            dq = np.full(L, 40 if ins[0] == ins[1] else 45)
            lines.append(" ".join([_noisy(rng, ref[o:o + L], 0.003), _phred(np.full(L, 30)),
                                   _phred(iq), _phred(dq), _phred(np.full(L, 10))]))
        haps = [ref, _noisy(rng, ref, 0.03)]
        text += "\n".join([f"{len(lines)} {len(haps)}"] + lines + haps) + "\n"
    b = G.HostBatch.parse(text)
    say(f"case: long reads' precision, semantics {semantics}, insertion qualities {ins}")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=semantics)
    low = ref < LOW
    assert low.sum() >= 40 and (~low).sum() >= 40 and ref.min() > -256
    for kw in ({}, {"small_batch": 0}):
        with G.Engine(semantics=semantics, **kw) as e:
            d = e.score_batch(b).astype(np.float64) - ref
        for part in (low, ~low):
            say(f"  mean {d[part].mean():.2e}, max {np.abs(d[part]).max():.2e}")
            assert abs(d[part].mean()) <= DRIFT
        half = 0.5 * np.spacing(np.abs(ref).astype(np.float32)).astype(np.float64)
        assert np.all(np.abs(d) <= half + PATH + DRIFT)


def _line(s, q, gap, gcp):
    L = len(s)
    gap = np.broadcast_to(gap, L)
    return " ".join([s, _phred(np.full(L, q)), _phred(gap), _phred(gap), _phred(np.full(L, gcp))])


def _check(lib, oracle, text, semantics):
    import gpupairhmm_amd as G
    b = G.HostBatch.parse(text)
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=semantics)
    for kw in ({}, {"small_batch": 0}, {"mode": G.MODE_PLAIN}):
        with G.Engine(semantics=semantics, **kw) as e:
            d = np.abs(e.score_batch(b).astype(np.float64) - ref)
        assert np.all(np.isfinite(d))
        # the parity bar, and a float's own step for scores in the thousands
        assert np.all(d <= 1e-3 + np.spacing(np.abs(ref).astype(np.float32))), (kw, ref[d > 1e-3])
    return ref


@pytest.mark.parametrize("semantics", [0, 1])
@pytest.mark.parametrize("L", [1024, 1031, 1032, 1200, 1535, 1536, 1537, 2047, 2048])
def test_long_gaps(lib, oracle, L, semantics):
    """A deletion or insertion of up to 400 bases between long flanks, whose run
    leaves the FP32 range within one row or column: by far the likeliest path
    all the same.  Lengths at the edges of tiles and lanes."""
    rng = np.random.default_rng(L)
    text = ""
    for k in (30, 75, 80, 100, 200, 400):
        ref, m = _seq(rng, L + 30), L // 2 + int(rng.integers(-200, 200))
        reads = [_line(ref[:L], 30, 40, 10),
                 _line((ref[:m] + _seq(rng, k) + ref[m:])[:L], 30, 40, 10),
                 _line(ref[:L], 20, rng.integers(25, 46, L), 12)]
        text += "\n".join([f"{len(reads)} 2"] + reads + [ref, ref[:m] + _seq(rng, k) + ref[m:]]) + "\n"
    say(f"case: long gaps, reads of {L}, semantics {semantics}")
    _check(lib, oracle, text, semantics)


@pytest.mark.parametrize("gcp", [6, 10, 25, 40, 60])
def test_scores_far_below(lib, oracle, gcp):
    """Scores down to thousands: reads hanging over either end of their hap,
    unrelated to it, or joined from two places of it in either order, so that a
    lane's values fall and rise again by far more than any scale holds."""
    rng = np.random.default_rng(gcp)
    text = ""
    for L in (1100, 1700):
        a, b = _seq(rng, L), _seq(rng, L)
        h = L // 2
        reads = [_line(s, 30, g, gcp) for g in (40, 30) for s in
                 (a, b[:h] + a[:L - h], a[h:] + a[:h], a[:h] + b[h:], _seq(rng, L))]
        haps = [a, a[:300], a[-400:], a[:h] + _seq(rng, 900) + a[h:], a[h:] + _seq(rng, 1000) + a[:h]]
        text += "\n".join([f"{len(reads)} {len(haps)}"] + reads + haps) + "\n"
    say(f"case: scores far below, gap continuation quality {gcp}")
    ref = _check(lib, oracle, text, 1)
    assert ref.min() < -1000 and ref.max() > -60


@pytest.mark.parametrize("semantics", [0, 1])
def test_padding_is_not_read(lib, semantics):
    """The bytes that pad a hap to whole dwords may be anything: one that is no
    base has no row in the emission tables, and the scores are the same bit for
    bit whatever stands there."""
    import gpupairhmm_amd as G
    rng = np.random.default_rng(71)
    text = ""
    for L in (60, 150, 1030, 1400):
        ref = _seq(rng, L + 40)
        reads = [_line(_noisy(rng, ref[o:o + L], 0.01), 30, 40, 10) for o in (0, 39)] + [
            _line(_seq(rng, L), 20, rng.integers(25, 46, L), 10)]
        haps = [ref[:n] for n in range(L + 37, L + 41)] + [_seq(rng, n) for n in (1, 2, 3, 62)]
        haps += [h[:20] + "N" + h[21:] for h in haps[:4]]
        text += "\n".join([f"{len(reads)} {len(haps)}"] + reads + haps) + "\n"
    b = G.HostBatch.parse(text)
    names = list(G._VIEW_ARRAYS)
    arrays = {k: np.array(b.array(k)) for k in names}
    within = np.zeros(len(arrays["hap_data"]), bool)
    for o, n in zip(arrays["hap_offsets"], arrays["hap_lengths"]):
        within[o:o + n] = True
    say(f"case: padding bytes, semantics {semantics}")
    want = {}
    for pad in (ord("N"), ord("A"), ord("T"), 0, 255):
        hap_data = np.where(within, arrays["hap_data"], np.uint8(pad))
        bb = G.HostBatch.from_arrays(**{**arrays, "hap_data": hap_data})
        for kw in ({}, {"small_batch": 0}, {"range_rescue": 0}):
            with G.Engine(semantics=semantics, **kw) as e:
                got = e.score_batch(bb).view(np.uint32)
            assert np.array_equal(got, want.setdefault(str(kw), got)), (pad, kw)


@pytest.mark.parametrize("small_batch", [0, 1 << 18])
def test_border_rows_are_as_long_as_the_strips_need(lib, oracle, small_batch):
    """A hap of four million bases, which only a read of 12 meets, leaves the
    scratch of an allocation-free call no border row of its length; the long
    reads, against haps of 1,300, need none like that."""
    import gpupairhmm_amd as G
    rng = np.random.default_rng(81)
    ref = _seq(rng, 1300)
    long_hap = rng.choice(np.frombuffer(b"ACGT", np.uint8), 4_000_000).tobytes().decode()
    text = "1 1\n" + _line(_seq(rng, 12), 30, 40, 10) + "\n" + long_hap + "\n"
    reads = [_line(_noisy(rng, ref[o:o + 1100], 0.01), 30, 40, 10) for o in range(0, 200, 10)]
    text += "\n".join([f"{len(reads)} 2"] + reads + [ref, _noisy(rng, ref, 0.02)]) + "\n"
    b = G.HostBatch.parse(text)
    say(f"case: border rows beside a very long hap, small_batch {small_batch}")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64)
    with G.Engine(small_batch=small_batch) as e:
        db, out = e.upload(b), e.alloc(4 * b.num_alignments)
        e.score_device_noalloc(db, out)
        e.synchronize()
        got = e.download(out, b.num_alignments)
        e.free(out)
        db.free()
    assert np.max(np.abs(got.astype(np.float64) - ref)) <= 1e-3


@pytest.mark.parametrize("small_batch", [0, 1 << 18])
def test_few_border_rows(lib, oracle, small_batch):
    """A long read against a hap of 60,000 bases leaves border rows for 260
    blocks; the strips share these, and the launch's other tasks, more than the
    blocks, are every block's: each is scored once, also a second time over
    another batch's scores."""
    import gpupairhmm_amd as G
    rng = np.random.default_rng(83)

    def batch():
        far = rng.choice(np.frombuffer(b"ACGT", np.uint8), 60_000).tobytes().decode()
        text = "1 1\n" + _line(far[:500] + far[700:1300], 30, 40, 10) + "\n" + far + "\n"
        ref = _seq(rng, 1300)
        reads = [_line(_noisy(rng, ref[o % 200:o % 200 + 1100], 0.01), 30, 40, 10) for o in range(400)]
        text += "\n".join([f"{len(reads)} 1"] + reads + [ref]) + "\n"
        ref = _seq(rng, 120)
        reads = [_line(_noisy(rng, ref[o % 60:o % 60 + 60], 0.01), 30, 40, 10) for o in range(90)]
        haps = [ref, ref[:70], ref[:40] + "N" + ref[41:]]
        text += ("\n".join([f"{len(reads)} {len(haps)}"] + reads + haps) + "\n") * 60
        return G.HostBatch.parse(text)

    b, other = batch(), batch()
    say(f"case: few border rows, small_batch {small_batch}, {b.num_alignments} alignments")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64)
    with G.Engine(small_batch=small_batch) as e:
        db, odb, out = e.upload(b), e.upload(other), e.alloc(4 * b.num_alignments)
        for x in (odb, db):
            e.score_device(x, out)
        e.synchronize()
        got = e.download(out, b.num_alignments)
        e.free(out)
        db.free()
        odb.free()
    assert np.max(np.abs(got.astype(np.float64) - ref)) <= 1e-3
