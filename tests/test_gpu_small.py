"""The few-launch sequence of small calls against plain mode, which sorts and
launches per class: the same bits, captured, eager, timed and allocation-free.
Records of one and of many reads and haps (more haps than the segment table
holds), empty reads and haps, every class of length, both arithmetic forms,
reads of several tiles, wildcard haps, bytes that match only themselves, scores
that the in-pass scaling refuses; and batches on either side of the limits on
records, alignments and columns.  The first batch is also compared with the
FP64 oracle.

Tolerance: the parity bar, 1e-3 absolute in log10 (FP32 sums of up to 1,600
rows and 1,700 columns: 3,300 roundings of 2^-24, 9e-5 in log10)."""
import numpy as np
import pytest

from conftest import say

pytestmark = pytest.mark.gpu

TOL = 1e-3


def _seq(rng, n, letters="ACGT"):
    return "".join(rng.choice(list(letters), n))


def _read(rng, haps, L, safe, exotic):
    hap = haps[int(rng.integers(len(haps)))]
    s = (hap[:L] + _seq(rng, max(0, L - len(hap)))) if rng.random() < 0.7 else _seq(rng, L)
    if exotic and L > 0 and rng.random() < 0.2:
        s = "R" + s[1:]
    q = rng.integers(2, 41, L)
    g = rng.integers(25, 46, L) if safe else np.full(L, 45)
    c = np.full(L, int(rng.integers(8, 15)))
    txt = [s] + ["".join(chr(33 + int(x)) for x in v) for v in (q, g, g, c)]
    return " ".join(txt)


def _record(rng, lens, haps, exotic=False):
    lines = [f"{len(lens)} {len(haps)}"]
    for L in lens:
        lines.append(_read(rng, haps, int(L), rng.random() < 0.5, exotic))
    return "\n".join(lines + haps) + "\n"


def _batches(name):
    rng = np.random.default_rng(23)
    if name == "shapes":
        t = _record(rng, [1], ["A"])
        t += _record(rng, rng.integers(1, 260, 90), [_seq(rng, int(n)) for n in rng.integers(1, 400, 7)])
        t += _record(rng, rng.integers(100, 1020, 20), [_seq(rng, int(n)) for n in rng.integers(5, 90, 150)])
        h = [_seq(rng, 300), _seq(rng, 211, "ACGTN"), _seq(rng, 64), "N", "ACGRT" * 9]
        t += _record(rng, rng.integers(1, 200, 40), h, exotic=True)
        t += _record(rng, [30, 1023, 1024, 1600, 800], [_seq(rng, 1700), _seq(rng, 500, "ACGTN")])
        return [t]
    if name == "records":  # the limit on records: 8192
        one = [_record(rng, rng.integers(1, 40, 2), [_seq(rng, 30)]) for _ in range(64)]
        return ["".join(one[i % 64] for i in range(n)) for n in (8191, 8192, 8193)]
    # the limits on alignments and columns
    one = [_record(rng, rng.integers(30, 120, 25), [_seq(rng, int(n)) for n in rng.integers(40, 90, 30)])
           for _ in range(16)]
    return ["".join(one[i % 16] for i in range(n)) for n in (87, 88, 349, 350)]


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("semantics", [0, 1])
@pytest.mark.parametrize("name", ["shapes", "records", "alignments"])
def test_small_calls(lib, oracle, name, semantics):
    import gpupairhmm_amd as G
    plain = G.Engine(semantics=semantics, mode=G.MODE_PLAIN)
    graph = G.Engine(semantics=semantics)
    eager = G.Engine(semantics=semantics, graphs=False)
    timed = G.Engine(semantics=semantics, time_kernels=True)
    for i, text in enumerate(_batches(name)):
        b = G.HostBatch.parse(text)
        say(f"case: {name} {i}, semantics {semantics}, {b.num_alignments} alignments")
        want = plain.score_batch(b)
        if i == 0:
            ref = oracle.score_batch(b.oracle_arrays(), oracle.F64, semantics=semantics)
            fin = np.isfinite(ref)
            assert (np.isfinite(want) == fin).all()
            assert np.max(np.abs(want[fin].astype(np.float64) - ref[fin])) <= TOL
        for e in (graph, eager, timed, graph):
            assert np.array_equal(_bits(e.score_batch(b)), _bits(want))
        db = graph.upload(b)
        out = graph.alloc(4 * b.num_alignments)
        for _ in range(3):
            graph.score_device(db, out)
        graph.score_device_noalloc(db, out)
        graph.synchronize()
        assert np.array_equal(_bits(graph.download(out, b.num_alignments)), _bits(want))
        graph.free(out)
        db.free()
    for e in (plain, graph, eager, timed):
        e.close()
