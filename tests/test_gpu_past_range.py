"""GPU test of pairs that pass the 16-bit range within a few columns (high match scores):
all of them are recomputed, also where their best lies on the last rows or columns, beside
padding whose values then mean nothing.  Every kernel form against the oracle."""
import numpy as np
import pytest

import oracle_lib as ol
import gbsw

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = gbsw.Context(0)
    yield c
    c.close()


def pairs(n, lo, hi, seed, letters):
    rng = np.random.default_rng(seed)
    refs, queries = [], []
    for _ in range(n):
        q_len = int(rng.integers(lo, hi + 1))
        r = letters[rng.integers(0, len(letters), int(rng.integers(1, 6 * q_len)))]
        at = int(rng.integers(0, len(r)))
        q = r[at:at + q_len].copy()  # often up to the end of r
        if len(q) < q_len:
            q = np.concatenate([q, letters[rng.integers(0, len(letters), q_len - len(q))]])
        change = rng.random(q_len) < rng.choice([0.0, 0.1, 0.5])
        q[change] = letters[rng.integers(0, len(letters), int(change.sum()))]
        if rng.random() < 0.5:
            r, q = q, r
        refs.append(r.tobytes())
        queries.append(q.tobytes())
    return gbsw.pack(refs) + gbsw.pack(queries)


def check(ctx, packed, scores, label):
    exp = ol.align_batch(*packed, ol.dna_scoring(*scores))
    b = ctx.batch(gbsw.DNA, *packed)
    try:
        b.align(gbsw.dna_scoring(*scores))
        got = b.results()
        for f in gbsw.FIELDS:
            bad = np.nonzero(got[f] != exp[f])[0]
            assert len(bad) == 0, "%s: %s differs at %d pairs, first %d: got %d want %d" % (
                label, f, len(bad), bad[0], got[f][bad[0]], exp[f][bad[0]])
        return {k["kind"] & 0xFF for k in b.launches()}
    finally:
        b.close()


@pytest.mark.parametrize("scores", [(4000, -1, -3, -40), (4000, -4000, -6, -1), (2000, -300, -40, -4), (1000, -100, -11, -2),
                                    (400, -300, -60, -30), (128, -128, -12, -2)])
@pytest.mark.parametrize("n,lo,hi,letters", [(3000, 1, 40, b"ACGTNWSKM"), (3000, 1, 40, b"ACGT"), (500, 30, 250, b"ACGT"),
                                             (60, 200, 900, b"ACGTN")])
def test_few_columns_past_the_range(ctx, scores, n, lo, hi, letters):
    packed = pairs(n, lo, hi, 0x5EED0730 + n + hi, np.frombuffer(letters, dtype=np.uint8))
    check(ctx, packed, scores, "%r, %d pairs" % (scores, n))


def test_two_pairs_that_were_missed(ctx):
    packed = gbsw.pack([b"@<=>=>?>"]) + gbsw.pack([b"?=?=AA?<>A@<>><A>>?>?=<==?=@A?><@<@><A?@?A@A<@A><<<?=?=>@?<?=@>=<=><?"])
    check(ctx, packed, (4000, -1, -3, -40), "eight columns")


@pytest.mark.parametrize("scores", [(224, -28, -10, -1), (192, -48, -12, -2)])
def test_eight_pairs_per_wave(ctx, scores):
    # byte tables: 16 columns of a lane gain up to 3,584
    packed = pairs(50000, 130, 180, 0x5EED0731, np.frombuffer(b"ACGT", dtype=np.uint8))
    ran = check(ctx, packed, scores, "%r" % (scores,))
    assert gbsw.KIND_BATCHED_PAIRS in ran, ran
