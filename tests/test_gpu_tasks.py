"""Copies of one record, from a launch with fewer tasks than waves to one with
many tasks per wave: every copy gets its score (none is left at that of the
other batch that was scored into the same output before), every copy the same
bits, and the first agrees with the FP64 oracle.  Each task of a launch must run exactly once wherever the waves take
their first one from.

Tolerance: the parity bar, 1e-3 absolute in log10 (reads of up to 40 rows:
about 100 roundings of 2^-24, 2.6e-6 in log10)."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

TOL = 1e-3


def _record(rng, lens, haps):
    lines = [f"{len(lens)} {len(haps)}"]
    for L in lens:
        seq = "".join(rng.choice(list("ACGT"), L))
        q = "".join(chr(33 + int(x)) for x in rng.integers(10, 41, L))
        g = chr(33 + 45) * L
        lines.append(" ".join([seq, q, g, g, chr(33 + 10) * L]))
    return "\n".join(lines + list(haps)) + "\n"


@pytest.mark.parametrize("copies", [1, 37, 500, 6000, 40000])
def test_every_copy_once(lib, oracle, copies):
    import gpupairhmm_amd as G
    rng = np.random.default_rng(17)
    haps = ["".join(rng.choice(list("ACGT"), n)) for n in (30, 61)]
    text = _record(rng, (9, 17, 31, 40), haps)
    one = G.HostBatch.parse(text)
    ref = oracle.score_batch(one.oracle_arrays(), oracle.F64, semantics=G.SEM_GPU)
    b = G.HostBatch.parse(text * copies)
    other = G.HostBatch.parse(_record(rng, (9, 17, 31, 40), haps) * copies)
    say(f"case: {copies} copies, {b.num_alignments} alignments")
    with G.Engine() as e:
        db = e.upload(b)
        out = e.alloc(4 * b.num_alignments)
        odb = e.upload(other)
        e.score_device(odb, out)
        e.score_device(db, out)
        e.synchronize()
        got = e.download(out, b.num_alignments).reshape(copies, -1)
        e.free(out)
        odb.free()
        db.free()
    assert np.isfinite(got).all()
    assert (got == got[0]).all()
    assert np.max(np.abs(got[0].astype(np.float64) - ref)) <= TOL


@pytest.mark.parametrize("small_batch", [0, 1 << 18])
@pytest.mark.parametrize("hap_len", [600, 120000])
def test_more_long_reads_than_border_rows(lib, oracle, small_batch, hap_len):
    """The longest hap of a batch sets the size of a border row, so one long
    hap leaves rows for 139 blocks only (256 MiB at 16 bytes a column): every
    long read must still be scored, also those after the last block's.  Reads
    of 1,030 rows against 600 columns: 1,630 roundings of 2^-24, 5e-5 in
    log10."""
    import gpupairhmm_amd as G
    rng = np.random.default_rng(29)
    text = _record(rng, (12,), ["".join(rng.choice(list("ACGT"), hap_len))])
    text += _record(rng, (1030,) * 300, ["".join(rng.choice(list("ACGT"), 600))])
    text += _record(rng, (40,) * 20, ["".join(rng.choice(list("ACGT"), 90)),
                                      "".join(rng.choice(list("ACGTN"), 90))])
    b = G.HostBatch.parse(text)
    say(f"case: hap {hap_len}, small_batch {small_batch}, {b.num_alignments} alignments")
    ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=G.SEM_GPU)
    with G.Engine(small_batch=small_batch) as e:
        got = e.score_batch(b)
    assert np.max(np.abs(got.astype(np.float64) - ref)) <= TOL
