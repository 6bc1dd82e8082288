"""Alignment paths at the edges of the path kernel's tiles and forms.

A wave's stripe has 16 K or 64 K columns (K <= 8); cells are 16-bit up to a value
bound of 7,936 or 16,384 and 32-bit above; scores are register tables (up to four
residue codes), byte profiles or word profiles (large or very negative scores).
Bar: the oracle's CIGAR words and path scores.
"""
import numpy as np
import pytest

import oracle_lib as ol
import gbsw
from gbsw import synth
from gbsw.scoring import BLOSUM62
from test_gpu_traceback import check_paths, pack

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = gbsw.Context(0)
    yield c
    c.close()


def related(rng, n, letters, subst=0.06, indels=2):
    """(ref, query): the query is the ref with substitutions and a few short gaps."""
    ref = rng.choice(letters, n)
    q = ref.copy()
    mut = rng.random(n) < subst
    q[mut] = rng.choice(letters, int(mut.sum()))
    for _ in range(indels if n > 40 else 0):
        at, k = int(rng.integers(5, len(q) - 20)), int(rng.integers(1, 9))
        if rng.random() < 0.5:
            q = np.delete(q, slice(at, at + k))
        else:
            q = np.insert(q, at, rng.choice(letters, k))
    return (ref.tobytes(), q.tobytes()) if rng.random() < 0.5 else (q.tobytes(), ref.tobytes())


EDGES = [1, 2, 3, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 66, 79, 80, 81, 95, 96, 97, 127, 128, 129, 130, 159,
         160, 161, 191, 192, 193, 255, 256, 257, 258, 319, 320, 321, 383, 384, 385, 511, 512, 513, 514, 640, 641]

# name, letters, scoring (match, mismatch, open, extend)
DNA_FORMS = [
    ("register tables", b"ACGT", (3, -3, -6, -1)),
    ("five codes, bytes", b"ACGTN", (3, -3, -6, -1)),
    ("equal gap costs", b"ACGT", (1, -1, -1, -1)),
    ("free extension", b"ACGT", (5, -4, -3, 0)),
    ("words, mismatch below a gap of each", b"ACGT", (2, -9, -3, -1)),
    ("words, wide 16-bit cells", b"ACGT", (20, -30, -60, -5)),
    ("32-bit cells", b"ACGT", (900, -700, -2000, -90)),
]


@pytest.mark.parametrize("name,letters,sc", DNA_FORMS, ids=[f[0] for f in DNA_FORMS])
def test_tile_edges(ctx, name, letters, sc):
    rng = np.random.default_rng(len(name))
    alpha = np.frombuffer(letters, np.uint8)
    pairs = [related(rng, n, alpha) for n in EDGES for _ in range(3)]
    rb, ro, qb, qo = pack(pairs)
    check_paths(ctx, gbsw.DNA, rb, ro, qb, qo, gbsw.dna_scoring(*sc), ol.dna_scoring(*sc), name)


@pytest.mark.parametrize("letters", [b"ACGT", b"ACGTN"])
def test_many_small_pairs(ctx, letters):
    # enough pairs for sixteen lanes per two pairs; unlike neighbours in a wave
    rng = np.random.default_rng(7)
    alpha = np.frombuffer(letters, np.uint8)
    pairs = [related(rng, int(rng.integers(1, 200)), alpha) for _ in range(30000)]
    rb, ro, qb, qo = pack(pairs)
    check_paths(ctx, gbsw.DNA, rb, ro, qb, qo, gbsw.dna_scoring(3, -3, -6, -1), ol.dna_scoring(3, -3, -6, -1),
                "small pairs %s" % letters.decode())


# value bound 3 n + 2 n + 19: around 7,936 and 16,384
@pytest.mark.parametrize("n", [1560, 1583, 1584, 1600, 3240, 3272, 3274, 3300])
def test_cell_range_edges(ctx, n):
    rng = np.random.default_rng(n)
    alpha = np.frombuffer(b"ACGT", np.uint8)
    same = rng.choice(alpha, n).tobytes()
    pairs = [(same, same)] + [related(rng, n, alpha, 0.02) for _ in range(3)] + [related(rng, 90, alpha)]
    rb, ro, qb, qo = pack(pairs)
    check_paths(ctx, gbsw.DNA, rb, ro, qb, qo, gbsw.dna_scoring(3, -3, -6, -1), ol.dna_scoring(3, -3, -6, -1),
                "identical %d" % n)


def test_protein_edges(ctx):
    rng = np.random.default_rng(5)
    alpha = np.frombuffer(b"ARNDCQEGHILKMFPSTWYV", np.uint8)
    pairs = [related(rng, n, alpha, 0.3) for n in EDGES for _ in range(3)]
    rb, ro, qb, qo = pack(pairs)
    for gaps in [(-6, -1), (-11, -1), (-2, -2)]:
        check_paths(ctx, gbsw.PROTEIN, rb, ro, qb, qo, gbsw.protein_scoring(BLOSUM62, *gaps),
                    ol.aa_scoring(BLOSUM62, *gaps), "protein %s" % (gaps,))


def test_flat_and_tall_rectangles(ctx):
    # extensions are free: a short sequence spreads over a long one, and a wave's
    # rectangles differ in shape far more than in area
    rng = np.random.default_rng(3)
    alpha = np.frombuffer(b"ACGT", np.uint8)
    pairs = []
    for k in range(120):
        long_, cut = rng.choice(alpha, int(rng.integers(600, 3000))), int(rng.integers(8, 40))
        short = np.concatenate([long_[:cut], long_[-cut:]])
        pairs.append((long_.tobytes(), short.tobytes()) if k % 2 else (short.tobytes(), long_.tobytes()))
    rb, ro, qb, qo = pack(pairs)
    check_paths(ctx, gbsw.DNA, rb, ro, qb, qo, gbsw.dna_scoring(5, -4, -3, 0), ol.dna_scoring(5, -4, -3, 0),
                "flat and tall")


def test_repeated_calls_reuse_the_scratch(ctx):
    w = synth.batched_dna(3000, seed=41)
    sc = gbsw.dna_scoring(*w.scoring)
    b = ctx.batch(gbsw.DNA, w.ref, w.ref_off, w.query, w.query_off)
    try:
        b.align(sc)
        first = b.traceback(sc)
        other = b.traceback(gbsw.dna_scoring(2, -9, -3, -1))  # other cells and forms
        again = b.traceback(sc)
    finally:
        b.close()
    assert len(other[0])
    for x, y in zip(first[:3], again[:3]):
        assert np.array_equal(x, y)
