"""The work order at the sizes where the preparing launch changes its way: up to
16,384 pairs sorted by one workgroup (1,024 threads, 16 pairs each), more by a radix
sort; one length for all pairs (one sort key) and every length class.  A pair left out
of the order, or in it twice at another's cost, keeps the cleared result."""
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


@pytest.mark.parametrize("n", [1, 2, 63, 1023, 1024, 1025, 2049, 16383, 16384, 16385])
@pytest.mark.parametrize("lengths", ["one", "mixed"])
def test_every_pair_is_aligned(ctx, n, lengths):
    rng = np.random.default_rng(n)
    L = np.frombuffer(b"ACGT", np.uint8)
    if lengths == "one":
        rl, ql = np.full(n, 24), np.full(n, 20)
    else:
        rl, ql = rng.integers(1, 80, n), rng.integers(1, 80, n)
        big = rng.integers(0, n, 6)  # a few of the far classes
        rl[big] = [300, 700, 1500, 9000, 200, 64][:len(big)]
        ql[big] = [280, 600, 1200, 2500, 5000, 640][:len(big)]
    ro = np.zeros(n + 1, np.uint64)
    qo = np.zeros(n + 1, np.uint64)
    np.cumsum(rl, out=ro[1:])
    np.cumsum(ql, out=qo[1:])
    rb, qb = L[rng.integers(0, 4, int(ro[-1]))], L[rng.integers(0, 4, int(qo[-1]))]
    exp = ol.align_batch(rb, ro, qb, qo, ol.dna_scoring(3, -3, -6, -1))
    sc = gbsw.dna_scoring(3, -3, -6, -1)
    b = ctx.batch(gbsw.DNA, rb, ro, qb, qo)
    try:
        for _ in range(3):  # recorded, then replayed
            b.align(sc)
            got = b.results()
            for f in gbsw.FIELDS:
                assert np.array_equal(exp[f], got[f]), (n, lengths, f)
    finally:
        b.close()
