"""GPU test of a serving slot with the least boundary rows a server takes and a scoring
outside the sweep kernels' range: long pairs of several classes that are admitted
together are answered (against the oracle), not refused."""
import numpy as np
import pytest

import oracle_lib as ol
import gbsw

pytestmark = pytest.mark.gpu

SCORES = (3, -3, -600, -600)


def test_long_pairs_of_several_classes_in_a_small_slot():
    rng = np.random.default_rng(0x5EED0702)
    bases = np.frombuffer(b"ACGT", dtype=np.uint8)
    refs, queries = [], []
    for rows, cols in ((60000, 300), (52000, 700), (64000, 1100), (58000, 420)):
        r = bases[rng.integers(0, 4, rows)]
        at = int(rng.integers(0, rows - cols))
        q = r[at:at + cols].copy()
        change = rng.random(cols) < 0.05
        q[change] = bases[rng.integers(0, 4, int(change.sum()))]
        refs.append(r.tobytes())
        queries.append(q.tobytes())
    packed = gbsw.pack(refs) + gbsw.pack(queries)
    exp = ol.align_batch(*packed, ol.dna_scoring(*SCORES))
    srv = gbsw.Server(0, slots=1, pairs_per_slot=64, residues_per_slot=1 << 20, boundary_bytes_per_slot=4 * 65000 * 4,
                      staging_bytes=1 << 20)
    try:
        ticket, out = srv.submit(gbsw.dna_scoring(*SCORES), *packed)
        info = srv.wait(ticket)
        assert info["status"] == 0
        for k, f in enumerate(gbsw.FIELDS):
            assert np.array_equal(out[k][:len(refs)], exp[f]), f
    finally:
        srv.close()
