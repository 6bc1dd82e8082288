"""GPU test of the sweep kernels with gap costs that do not fit the byte tables together
with the scores (gaps that cost nothing or little, and dear ones: the tables then hold the
scores from the smallest up, and the step adds the rest), and with gaps so dear that the
running offset takes most of the 16-bit range.  Every kernel form against the oracle, and
jobs just below and above the limit of the range."""
import numpy as np
import pytest

import oracle_lib as ol
import gbsw
from gbsw import synth
from gbsw.scoring import BLOSUM62

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = gbsw.Context(0)
    yield c
    c.close()


def compare(ctx, packed, gsc, osc, label, paths=True):
    exp = ol.align_batch(*packed, osc)
    b = ctx.batch(gsc.alphabet, *packed)
    try:
        b.align(gsc)
        got = b.results()
        for f in gbsw.FIELDS:
            bad = np.nonzero(got[f] != exp[f])[0]
            assert len(bad) == 0, "%s: %s differs at %d pairs, first %d: got %d want %d" % (
                label, f, len(bad), bad[0], got[f][bad[0]], exp[f][bad[0]])
        ran = {k["kind"] & 0xFF for k in b.launches()}
        # alignment paths too, where a run of gaps is one gap
        if paths and gsc.gap_open <= gsc.gap_extend:
            words, off, ps, _ = b.traceback(gsc)
            ew, eoff, eps = ol.traceback_batch(*packed, osc, exp)
            assert np.array_equal(words, ew) and np.array_equal(off, eoff) and np.array_equal(ps, eps), label
        return ran
    finally:
        b.close()


def reads(n, lo, hi, seed, alphabet=b"ACGT", spread=3.0):
    rng = np.random.default_rng(seed)
    letters = np.frombuffer(alphabet, dtype=np.uint8)
    refs, queries = [], []
    for _ in range(n):
        q_len = int(rng.integers(lo, hi + 1))
        r = letters[rng.integers(0, len(letters), int(q_len + rng.integers(0, max(1, int(spread * q_len)))))]
        at = int(rng.integers(0, len(r) - q_len + 1))
        q = r[at:at + q_len].copy()
        change = rng.random(q_len) < 0.1
        q[change] = letters[rng.integers(0, len(letters), int(change.sum()))]
        cut = int(rng.integers(0, q_len))
        refs.append(r.tobytes())
        queries.append(np.delete(q, cut).tobytes() if q_len > 3 and rng.random() < 0.5 else q.tobytes())
    return gbsw.pack(refs) + gbsw.pack(queries)


DNA = [(3, -3, 0, 0), (1, 0, 0, 0), (2, -1, 0, 0), (3, -3, 0, -4), (3, -3, -4, 0), (3, -3, -600, -100), (10, -10, -60, -50),
       (1, -1, -8000, -20), (2, -3, -50, -140)]


@pytest.mark.parametrize("scores", DNA)
@pytest.mark.parametrize("n,lo,hi", [(1, 1, 40), (9, 500, 1500), (300, 1, 700), (2500, 20, 250), (40, 900, 1100)])
def test_dna(ctx, scores, n, lo, hi):
    packed = reads(n, lo, hi, 0x5EED0720 + n)
    ran = compare(ctx, packed, gbsw.dna_scoring(*scores), ol.dna_scoring(*scores), "%r n %d" % (scores, n))
    assert ran <= {gbsw.KIND_BATCHED_F16, gbsw.KIND_SPLIT_F16}, ran


@pytest.mark.parametrize("gaps", [(0, 0), (-300, -90), (0, -3)])
@pytest.mark.parametrize("swap", [False, True])
def test_protein(ctx, gaps, swap):
    w = synth.plain_protein(300, seed=0x5EED0721)
    table = list(BLOSUM62)
    if swap: # an asymmetric table
        table[0 * 24 + 1], table[3 * 24 + 7] = 2, -5
    packed = (w.ref, w.ref_off, w.query, w.query_off)
    ran = compare(ctx, packed, gbsw.protein_scoring(table, *gaps), ol.aa_scoring(table, *gaps), "%r %r" % (gaps, swap))
    assert ran <= {gbsw.KIND_BATCHED_F16, gbsw.KIND_SPLIT_F16}, ran


@pytest.mark.parametrize("scores", [(3, -3, 0, 0), (3, -3, -600, -100), (1, -3, -1, -1)])
@pytest.mark.parametrize("n,lo,hi,kind", [(40000, 8, 120, "pairs"), (80000, 130, 256, "pairs"), (9000, 257, 400, "four")])
def test_many_reads(ctx, scores, n, lo, hi, kind):
    # eight pairs per wave, narrow and wide geometries; four pairs per wave, wide ones
    packed = reads(n, lo, hi, 0x5EED0723, spread=0.1)
    ran = compare(ctx, packed, gbsw.dna_scoring(*scores), ol.dna_scoring(*scores), "%r n %d" % (scores, n), paths=False)
    assert (gbsw.KIND_BATCHED_PAIRS if kind == "pairs" else gbsw.KIND_BATCHED_F16) in ran, ran


@pytest.mark.parametrize("n,lo,hi", [(3000, 20, 250), (20000, 257, 400)])
def test_many_proteins(ctx, n, lo, hi):
    # four pairs per wave, byte profile, narrow and wide geometries
    packed = reads(n, lo, hi, 0x5EED0724, alphabet=b"ARNDCQEGHILKMFPSTWYV", spread=0.1)
    ran = compare(ctx, packed, gbsw.protein_scoring(BLOSUM62, -2, -1), ol.aa_scoring(BLOSUM62, -2, -1), "proteins %d" % n,
                  paths=False)
    assert gbsw.KIND_BATCHED_F16 in ran, ran


def test_at_the_limit_of_the_range(ctx):
    # -140 per gap position: the offset leaves 5,783 of the 16-bit range
    # (0x7C00 - 2048 - 23,624 - 280 - 9), which 1,150 identical columns at +5 stay
    # under and 1,165 do not: those take the int16 kernels
    rng = np.random.default_rng(0x5EED0722)
    bases = np.frombuffer(b"ACGT", dtype=np.uint8)
    sc = (5, -4, -100, -140)
    for cols, sweeps in ((1150, True), (1165, False)):
        seqs = [bases[rng.integers(0, 4, c)].tobytes() for c in (cols, cols, cols // 2, 33, 64)]
        packed = gbsw.pack([s + b"ACGT" for s in seqs]) + gbsw.pack(seqs)
        ran = compare(ctx, packed, gbsw.dna_scoring(*sc), ol.dna_scoring(*sc), "%d columns" % cols)
        assert (ran <= {gbsw.KIND_BATCHED_F16, gbsw.KIND_SPLIT_F16}) == sweeps, (cols, ran)
