"""GPU test of a launch whose geometry changes from class to class: seventeen pairs of
seventeen geometry ranges (without the split form) against the oracle, in a resident
batch, in one call and in a serving slot."""
import numpy as np
import pytest

import oracle_lib as ol
import gbsw

pytestmark = pytest.mark.gpu

# (longer, shorter), as kUnsplitRanges of host/plan_check.cpp
LENGTHS = [(5642, 5151), (5633, 5633), (4631, 4631), (4151, 4151), (3680, 3680), (3087, 3087), (2574, 2574),
           (2049, 2049), (1543, 1543), (1033, 1033), (778, 778), (647, 647), (514, 514), (386, 386), (257, 257),
           (130, 130), (20, 20)]
SCORES = (3, -3, -6, -1)


@pytest.fixture(scope="module")
def pairs():
    rng = np.random.default_rng(0x5EED0701)
    bases = np.frombuffer(b"ACGT", dtype=np.uint8)
    refs, queries = [], []
    for rows, cols in LENGTHS:
        r = bases[rng.integers(0, 4, rows)]
        q = r[:cols].copy()
        change = rng.random(cols) < 0.1
        q[change] = bases[rng.integers(0, 4, int(change.sum()))]
        refs.append(r.tobytes())
        queries.append(q.tobytes())
    packed = gbsw.pack(refs) + gbsw.pack(queries)
    return packed, ol.align_batch(*packed, ol.dna_scoring(*SCORES))


def check(got, exp, label):
    for f in gbsw.FIELDS:
        bad = np.nonzero(got[f] != exp[f])[0]
        assert len(bad) == 0, "%s: %s differs at pairs %s" % (label, f, [LENGTHS[k] for k in bad])


def test_batch_and_call(pairs):
    packed, exp = pairs
    ctx = gbsw.Context(0)
    try:
        ctx.set_option(gbsw.OPT_SPLIT, 0)
        sc = gbsw.dna_scoring(*SCORES)
        b = ctx.batch(gbsw.DNA, *packed)
        for turn in range(3): # captured, then replayed
            b.align(sc)
            check(b.results(), exp, "batch, turn %d" % turn)
        assert [(k["kind"] & 0xFF, k["pairs"]) for k in b.launches()] == [(gbsw.KIND_BATCHED_F16, len(LENGTHS))]
        b.close()
        check(ctx.align_packed(*packed, sc), exp, "call")
        check(ctx.align_packed(*packed, sc, noalloc=True), exp, "allocation-free call")
    finally:
        ctx.close()


def test_serving_slot(pairs, monkeypatch):
    packed, exp = pairs
    monkeypatch.setenv("GBSW_SPLIT", "0")
    srv = gbsw.Server(0, slots=1, pairs_per_slot=256, residues_per_slot=1 << 20, boundary_bytes_per_slot=64 << 20,
                      staging_bytes=1 << 20)
    try:
        ticket, out = srv.submit(gbsw.dna_scoring(*SCORES), *packed)
        srv.wait(ticket)
        check(dict(zip(gbsw.FIELDS, out[:, :len(LENGTHS)])), exp, "serving slot")
    finally:
        srv.close()
