"""Reads of several tiles (strips) and haps holding the wildcard, against the
FP64 oracle and against the one-wave kernel that takes them when the FP32 pass
does not scale (range_rescue 0): lengths around the strips' tiles of 768 rows,
reads hanging over their hap, both arithmetic forms, both per-read semantics,
the wildcard on either path, and runs of items that do not fill a wave.

Tolerance: the parity bar, 1e-3 absolute in log10.  FP32 sums of up to 2,400
rows and 2,500 columns of positive terms are good to about 5,000 roundings of
2^-24, 3e-4 relative or 1.3e-4 in log10, whatever the score."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

TOL = 1e-3


def _record(reads, haps):
    lines = [f"{len(reads)} {len(haps)}"]
    for r, bq, gap, gcp in reads:
        q = "".join(chr(33 + int(x)) for x in bq)
        g = "".join(chr(33 + int(x)) for x in gap)
        c = "".join(chr(33 + int(x)) for x in gcp)
        lines.append(" ".join([r, q, g, g, c]))
    return "\n".join(lines + list(haps)) + "\n"


def _seq(rng, n):
    return "".join(rng.choice(list("ACGT"), n))


def _noisy(rng, s, err):
    s = list(s)
    for i in np.flatnonzero(rng.random(len(s)) < err):
        s[i] = "ACGT"[int(rng.integers(4))]
    return "".join(s)


def _read(rng, seq, form):
    L = len(seq)
    gap = np.full(L, 40) if form == "fast" else rng.integers(25, 46, L)
    return seq, rng.integers(10, 41, L), gap, np.full(L, int(rng.integers(8, 15)))


def _max_delta(got, ref):
    return float(np.max(np.abs(np.asarray(got, np.float64) - ref)))


def _check(lib, oracle, text, semantics, name):
    import gpupairhmm_amd as G
    b = G.HostBatch.parse(text)
    say(f"case: {name}, semantics {semantics}, {b.num_alignments} alignments")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=semantics)
    with G.Engine(semantics=semantics) as e:
        got = e.score_batch(b)
    with G.Engine(semantics=semantics, mode=G.MODE_PLAIN) as e:
        plain = e.score_batch(b)
    with G.Engine(semantics=semantics, range_rescue=False) as e:
        one_wave = e.score_batch(b)
    assert np.all(np.isfinite(got))
    assert _max_delta(got, ref) <= TOL
    assert _max_delta(one_wave, ref) <= TOL
    assert np.array_equal(got.view(np.uint32), plain.view(np.uint32))


@pytest.mark.parametrize("semantics", [0, 1])
@pytest.mark.parametrize("form", ["fast", "safe"])
def test_strips(lib, oracle, form, semantics):
    """Reads of one row more than the largest tile up to four strips, from
    their hap, longer than it at either end, and unrelated to it."""
    rng = np.random.default_rng(91)
    text = ""
    for L in (1024, 1535, 1536, 1537, 1551, 2303, 2304, 2305):
        ref = _seq(rng, L + 60)
        reads = [_read(rng, _noisy(rng, ref[20:20 + L], 0.01), form),
                 _read(rng, _noisy(rng, ref[60:60 + L], 0.02), form),
                 _read(rng, _seq(rng, L), form)]
        haps = [ref, ref[:L - 40], ref[90:], _seq(rng, 17), _seq(rng, 700)]
        text += _record(reads, haps)
    _check(lib, oracle, text, semantics, f"strips, {form}")


@pytest.mark.parametrize("semantics", [0, 1])
def test_wildcard_haps(lib, oracle, semantics):
    """Haps with runs of N anywhere: reads of 1 to 1023 bases from them (and
    longer ones on strips), so that a wave holds from 1 to 24 items."""
    rng = np.random.default_rng(92)
    text = ""
    for L in (1, 15, 16, 31, 47, 100, 167, 168, 335, 336, 511, 512, 1007, 1008, 1023, 1100, 1600):
        ref = _seq(rng, L + 90)
        haps = []
        for at in (0, 45 + L // 2, L + 85):
            h = list(ref)
            h[at:at + 5] = "N" * len(h[at:at + 5])
            haps.append("".join(h))
        haps.append(ref)
        n = 27 if L < 200 else 3
        reads = [_read(rng, _noisy(rng, ref[o:o + L], 0.01), ("fast", "safe")[i % 2])
                 for i, o in enumerate(rng.integers(0, 90, n))]
        text += _record(reads, haps)
    _check(lib, oracle, text, semantics, "wildcard haps")


def test_wildcard_haps_far_below_the_fp32_range(lib, oracle):
    """Unrelated reads and haps with a wildcard, scores below -100: the packed
    FP64 pass, with reads on either side of its 512 rows."""
    rng = np.random.default_rng(93)
    text = ""
    for L in (150, 167, 168, 300, 510, 511, 512, 900):
        reads = [_read(rng, _seq(rng, L), ("fast", "safe")[i % 2]) for i in range(5)]
        haps = []
        for H in (L // 2, L + 100, L + 150):
            h = list(_seq(rng, H))
            h[H // 3] = "N"
            haps.append("".join(h))
        text += _record(reads, haps)
    _check(lib, oracle, text, 0, "wildcard haps, low scores")
