"""Haps holding the wildcard, or a byte that matches nothing but itself, under
reads that hang over an end of them: the sum is complete at the hap's last
column, and stays what it is there, whatever the sweep's other lanes still
compute past it.

Tolerance: the parity bar, 1e-3 absolute in log10 (FP32 sums of up to 1,100 rows
of positive terms are good to about 2,200 roundings of 2^-24, 1.3e-4 relative or
6e-5 in log10)."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

TOL = 1e-3


def _seq(rng, n):
    return "".join(rng.choice(list("ACGT"), n))


def _phred(q):
    return "".join(chr(33 + int(x)) for x in q)


def _overhanging(rng, byte):
    """Records of reads of which 40 to 90 bases lie past their hap's end, or
    before its start, each hap with one `byte` in it; one within its hap."""
    text = ""
    for L in (100, 150, 167, 168, 300, 511, 512, 900, 1100):
        ref = _seq(rng, L + 200)
        hap = ref[100:100 + L]
        lines = []
        for o in [100 + n for n in range(40, 91, 2)] + [100 - n for n in range(40, 91, 10)] + [100]:
            q = rng.integers(25, 41, L)
            lines.append(" ".join([ref[o:o + L], _phred(q), _phred(np.full(L, 40)),
                                   _phred(np.full(L, 40)), _phred(np.full(L, 10))]))
        haps = [hap[:at] + byte + hap[at + 1:] for at in (3, L // 2, L - 2)]
        text += "\n".join([f"{len(lines)} {len(haps)}"] + lines + haps) + "\n"
    return text


@pytest.mark.parametrize("semantics", [0, 1, 2])
@pytest.mark.parametrize("byte", ["N", "R"])
def test_reads_past_the_hap(lib, oracle, byte, semantics):
    import gpupairhmm_amd as G
    b = G.HostBatch.parse(_overhanging(np.random.default_rng(95), byte))
    say(f"case: reads past haps with {byte}, semantics {semantics}, {b.num_alignments} alignments")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=semantics)
    assert np.count_nonzero((ref > -80) & (ref < -60)) >= 100
    for kw in ({}, {"small_batch": 0}, {"mode": G.MODE_PLAIN}, {"range_rescue": 0}):
        with G.Engine(semantics=semantics, **kw) as e:
            d = np.abs(e.score_batch(b).astype(np.float64) - ref)
        say(f"  {kw}: max {np.nanmax(d):.2e}, {np.count_nonzero(~(d <= TOL))} off")
        assert np.all(d <= TOL), (kw, ref[~(d <= TOL)])
