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
