"""Inputs at the sizes where the upload changes its way: one staged block up to 1 MiB,
plain copies up to 8 MiB, several threads and a ring of pinned pieces above; residues
scanned on the host up to 64 KiB; results behind the kernels up to 16,384 pairs.  The
allocation-free entry point copies plainly at every size: all five outputs equal its."""
import threading

import numpy as np
import pytest

import gbsw

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = gbsw.Context(0)
    yield c
    c.close()


def make(seed, total, per_pair, letters=b"ACGTN"):
    rng = np.random.default_rng(seed)
    n = max(1, total // per_pair)
    ql = rng.integers(1, per_pair // 2 + 1, n)
    rl = per_pair - ql
    rl[0] += max(0, total - int(rl.sum() + ql.sum()))  # exactly `total` residues
    if rl[0] > 60000:
        rl[0] = 60000
    ro = np.zeros(n + 1, np.uint64)
    qo = np.zeros(n + 1, np.uint64)
    np.cumsum(rl, out=ro[1:])
    np.cumsum(ql, out=qo[1:])
    L = np.frombuffer(letters, np.uint8)
    rb, qb = L[rng.integers(0, len(L) - 1, int(ro[-1]))], L[rng.integers(0, len(L) - 1, int(qo[-1]))]
    qb[-1] = L[-1]  # a code only the last byte shows
    return rb, ro, qb, qo


SIZES = [(2, 2), (300, 300), (65535, 120), (65536, 120), (65537, 120), (900_000, 300), (1_040_000, 300), (2_000_003, 90),
         (7_900_000, 400), (8_600_000, 400), (24_000_001, 500)]


@pytest.mark.parametrize("total,per_pair", SIZES)
def test_equal_to_plain_copies(ctx, total, per_pair):
    w = make(total, total, per_pair)
    sc = gbsw.dna_scoring(3, -3, -6, -1)
    exp = ctx.align_packed(*w, sc, noalloc=True)
    for _ in range(2):
        got = ctx.align_packed(*w, sc)
        for f in gbsw.FIELDS:
            assert np.array_equal(exp[f], got[f]), (total, f)
    b = ctx.batch(gbsw.DNA, *w)
    try:
        b.align(sc)
        got = b.results()
    finally:
        b.close()
    for f in gbsw.FIELDS:
        assert np.array_equal(exp[f], got[f]), (total, f)


def test_batches_from_several_threads(ctx):
    # one context's batches share the ring
    ws = [make(s, 9_000_000, 300) for s in range(3)]
    got = [None] * 3

    def create(k):
        got[k] = ctx.batch(gbsw.DNA, *ws[k])

    ts = [threading.Thread(target=create, args=(k,)) for k in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    sc = gbsw.dna_scoring(3, -3, -6, -1)
    for k in range(3):
        exp = ctx.align_packed(*ws[k], sc, noalloc=True)
        got[k].align(sc)
        res = got[k].results()
        got[k].close()
        for f in gbsw.FIELDS:
            assert np.array_equal(exp[f], res[f]), (k, f)
