"""The sweep kernels (batched form) against the oracle at the sizes where they can
go wrong: column counts around a lane block, a strip and a wave; row counts around
a chunk, the period of the running offset and a group's fill; every profile form;
and scores around the top of the 16-bit range.  Bit-exact on all five outputs;
the int16 kernels (option F16 off) must agree on the same pairs."""
import random

import numpy as np
import pytest

import oracle_lib as ol
import gbsw
from gbsw.scoring import AA_ORDER, BLOSUM62

pytestmark = pytest.mark.gpu
FIELDS = gbsw.FIELDS


@pytest.fixture(scope="module")
def ctx():
    c = gbsw.Context(0)
    yield c
    c.close()


def mutate(rng, s, letters):
    out = []
    for c in s:
        u = rng.random()
        if u < 0.08:
            out.append(rng.choice(letters))
        elif u < 0.10:
            continue
        elif u < 0.12:
            out.append(c + rng.choice(letters))
        else:
            out.append(c)
    return "".join(out)


def edge_pairs(seed, letters, cols, rows):
    rng = random.Random(seed)
    refs, qrys = [], []
    for c in cols:
        for r in rows:
            long, short = max(c, r), min(c, r)
            a = "".join(rng.choice(letters) for _ in range(long))
            at = rng.randint(0, long - short)
            b = mutate(rng, a[at:at + short], letters) if rng.random() < 0.7 else \
                "".join(rng.choice(letters) for _ in range(short))
            b = (b + "".join(rng.choice(letters) for _ in range(short)))[:short]
            refs.append(a)
            qrys.append(b)
            if rng.random() < 0.3:
                refs[-1], qrys[-1] = qrys[-1], refs[-1]
    return refs, qrys


def check(ctx, refs, qrys, oracle_sc, sc, label):
    rb, ro = gbsw.pack(refs)
    qb, qo = gbsw.pack(qrys)
    exp = ol.align_batch(rb, ro, qb, qo, oracle_sc)
    try:
        for f16, split in ((1, 1), (1, 0), (0, 0)):
            print("case", label, "f16", f16, "split", split, flush=True)
            ctx.set_option(gbsw.OPT_F16, f16)
            ctx.set_option(gbsw.OPT_SPLIT, split)
            got = ctx.align_packed(rb, ro, qb, qo, sc, "batched")
            for f in FIELDS:
                bad = np.nonzero(got[f] != exp[f])[0]
                assert len(bad) == 0, (label, f16, split, f, len(bad), int(bad[0]), len(refs[bad[0]]),
                                       len(qrys[bad[0]]), {g: (int(got[g][bad[0]]), int(exp[g][bad[0]])) for g in FIELDS})
    finally:
        ctx.set_option(gbsw.OPT_F16, 1)
        ctx.set_option(gbsw.OPT_SPLIT, 1)
    return exp


COLS = (1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 159, 160, 161, 255, 256, 257, 383, 385, 511, 512, 513, 1025)
ROWS = (1, 16, 32, 97, 128, 129, 161, 225, 256, 257, 289, 600, 1200)
DNA_FORMS = [("ACGT", (3, -3, -6, -1)),       # register tables
             ("ACG", (1, -4, -6, 0)),         # no extension cost: no running offset
             ("ACGT", (4, -4, -40, -24)),     # a large one
             ("ACGTN", (3, -3, -6, -1)),      # byte profile
             ("ACGTNRYKMSWB", (2, -3, -5, -2)),
             ("ACGT", (9, -11, -13, -2)),     # 16-bit profile
             ("ACGT", (2, -200, -6, -1)),     # 16-bit, negative after the bias
             ("ACGT", (3, -3, -1, -4)),       # extending costs more than opening
             ("ACGT", (3, -3, -600, -600))]   # outside the sweep kernels' range


@pytest.mark.parametrize("form", range(len(DNA_FORMS)))
def test_dna_tile_edges(ctx, form):
    letters, scoring = DNA_FORMS[form]
    refs, qrys = edge_pairs(900 + form, letters, COLS, ROWS)
    check(ctx, refs, qrys, ol.dna_scoring(*scoring), gbsw.dna_scoring(*scoring), "dna %s %s" % (letters, scoring))


@pytest.mark.parametrize("gaps", [(-6, -1), (-11, -1), (-1, -1), (0, 0)])
def test_protein_tile_edges(ctx, gaps):
    refs, qrys = edge_pairs(950 - gaps[0], AA_ORDER[:20], COLS, ROWS)
    check(ctx, refs, qrys, ol.aa_scoring(BLOSUM62, *gaps), gbsw.protein_scoring(BLOSUM62, *gaps), "protein %s" % (gaps,))


@pytest.mark.parametrize("letters", ["ACGT", "ACGTN"])
def test_scores_around_the_16_bit_range(ctx, letters):
    """Identical stretches of 96 per residue: scores from 30,000 to 34,000 cross the
    limit from which a pair is recomputed with int32 cells, beside ordinary pairs."""
    rng = random.Random(77)
    refs, qrys = [], []
    for n in list(range(312, 356)) + [900, 1500]:
        core = "".join(rng.choice(letters) for _ in range(n))
        refs.append("".join(rng.choice(letters) for _ in range(rng.randint(0, 200))) + core)
        qrys.append(core)
        refs.append("".join(rng.choice(letters) for _ in range(400)))
        qrys.append(refs[-1][100:100 + rng.randint(1, 120)])
    exp = check(ctx, refs, qrys, ol.dna_scoring(96, -96, -192, -64), gbsw.dna_scoring(96, -96, -192, -64), letters)
    assert exp["score"].max() > 100_000 and ((exp["score"] > 30_000) & (exp["score"] < 33_000)).sum() > 10


PAIRS = 120000  # enough pairs of up to 256 columns for eight per wave (16 lanes for two)


@pytest.mark.parametrize("letters,sc", [("ACGT", (3, -3, -6, -1)), ("ACG", (1, -1, -1, -1)), ("ACGT", (112, -16, -32, -2))])
def test_eight_pairs_per_wave(ctx, letters, sc):
    # columns around every multiple of 16, rows around a chunk and a ring; equal lengths
    # (the reverse pass may swap the sequences), pairs past the 16-bit range, no score
    rng = np.random.default_rng(len(letters) + sc[0])
    L = np.frombuffer(letters.encode(), np.uint8)
    edge = np.array([c + d for c in range(16, 257, 16) for d in (-1, 0, 1)])
    cols = np.where(rng.random(PAIRS) < 0.5, rng.choice(edge[edge <= 256], PAIRS), rng.integers(1, 257, PAIRS))
    cols[rng.random(PAIRS) < 0.7] //= 3
    cols = np.maximum(cols, 1)
    rows = cols + rng.choice([0, 1, 15, 31, 32, 33, 63, 64, 65, 130], PAIRS)
    refs, qrys = [], []
    for c, r in zip(cols, rows):
        a = L[rng.integers(0, len(L), r)]
        at = int(rng.integers(0, r - c + 1))
        b = a[at:at + c].copy()
        u = rng.random()
        if u < 0.25:
            b = L[rng.integers(0, len(L), c)]
        elif u < 0.8:
            hit = rng.random(c) < 0.1
            b[hit] = L[rng.integers(0, len(L), int(hit.sum()))]
            if c > 20 and u < 0.5:  # a short gap
                k = int(rng.integers(1, 6))
                b = np.concatenate([b[:c // 2], b[c // 2 + k:], L[rng.integers(0, len(L), k)]])
        x, y = a.tobytes(), b.tobytes()
        refs.append(x if rng.random() < 0.7 else y)
        qrys.append(y if refs[-1] is x else x)
    refs[5], qrys[5] = b"A" * 60, b"C" * 40
    ro = np.zeros(PAIRS + 1, np.uint64)
    qo = np.zeros(PAIRS + 1, np.uint64)
    np.cumsum([len(x) for x in refs], out=ro[1:])
    np.cumsum([len(x) for x in qrys], out=qo[1:])
    rb, qb = np.frombuffer(b"".join(refs), np.uint8), np.frombuffer(b"".join(qrys), np.uint8)
    exp = ol.align_batch(rb, ro, qb, qo, ol.dna_scoring(*sc))
    b = ctx.batch(gbsw.DNA, rb, ro, qb, qo)
    try:
        b.align(gbsw.dna_scoring(*sc))
        got, launches = b.results(), b.launches()
    finally:
        b.close()
    # columns per lane of 16 lanes, not of two blocks of 16
    assert max(x["columns_per_lane"] for x in launches if x["pairs"] > 1000) == 16, launches
    for f in FIELDS:
        bad = np.nonzero(exp[f] != got[f])[0]
        assert len(bad) == 0, (sc, f, len(bad), refs[bad[0]], qrys[bad[0]], exp[f][bad[0]], got[f][bad[0]])


def test_long_pairs_take_int32_cells_at_once(ctx):
    # a class whose longest pair may pass the 16-bit range runs on int32 cells beside the
    # rest: one pair that passes it, an unrelated one of its class, shorter ones, and one
    # that passes it from a shorter class (no errors: recomputed after the rest)
    rng = np.random.default_rng(77)
    L = np.frombuffer(b"ACGT", np.uint8)

    def related(n, subst):
        a = L[rng.integers(0, 4, n)]
        b = a.copy()
        hit = rng.random(n) < subst
        b[hit] = L[rng.integers(0, 4, int(hit.sum()))]
        return a.tobytes(), np.delete(b, slice(n // 3, n // 3 + 7)).tobytes()

    pairs = [related(13400, 0.08), (L[rng.integers(0, 4, 13500)].tobytes(), L[rng.integers(0, 4, 13350)].tobytes()),
             related(10300, 0.0)] + [related(int(n), 0.1) for n in rng.integers(200, 3000, 30)]
    rb, ro = gbsw.pack([p[0] for p in pairs])
    qb, qo = gbsw.pack([p[1] for p in pairs])
    exp = ol.align_batch(rb, ro, qb, qo, ol.dna_scoring(3, -3, -6, -1))
    assert exp["score"][0] > 29000 and exp["score"][2] > 29000 and exp["score"][1] < 28000
    sc = gbsw.dna_scoring(3, -3, -6, -1)
    b = ctx.batch(gbsw.DNA, rb, ro, qb, qo)
    try:
        for split in (1, 0):  # without the split form every such pair is recomputed
            ctx.set_option(gbsw.OPT_SPLIT, split)
            for _ in range(2):
                b.align(sc)
                got, wide = b.results(), [x["pairs"] for x in b.launches() if x["kind"] == 3]
                assert wide == ([2, 1] if split else [2]), wide
                for f in FIELDS:
                    assert np.array_equal(exp[f], got[f]), (split, f)
    finally:
        ctx.set_option(gbsw.OPT_SPLIT, 1)
        b.close()
