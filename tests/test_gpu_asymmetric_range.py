"""GPU test of asymmetric tables whose reversed boxes score past the 16-bit range while
the forward pass stays below it: such pairs are recomputed, and the job is not reported
as failed.  Against the oracle, in both forms and in one call."""
import random

import numpy as np
import pytest

import oracle_lib as ol
import gbsw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gaps", [(-5, -90), (-9000, -90), (-5, -2)])
@pytest.mark.parametrize("most,seed", [(3000, 1), (900, 2), (8000, 3)])
def test_reversed_boxes_past_the_range(gaps, most, seed):
    rng = random.Random(0x5EED0740 + seed)
    table = [rng.randint(-most, most) for _ in range(576)]
    letters = "ARNDCQEGHILKMFPSTWYVBZX*"
    refs, queries = [], []
    for _ in range(1500):
        a = "".join(rng.choice(letters) for _ in range(rng.randint(5, 60)))
        b = "".join(rng.choice(letters) for _ in range(rng.randint(5, 60)))
        refs.append(a)
        queries.append(a[:len(b)] if rng.random() < 0.5 else b)
    packed = gbsw.pack(refs) + gbsw.pack(queries)
    exp = ol.align_batch(*packed, ol.aa_scoring(table, *gaps))
    sc = gbsw.protein_scoring(table, *gaps)
    ctx = gbsw.Context(0)
    try:
        b = ctx.batch(gbsw.PROTEIN, *packed)
        got = [ctx.align_packed(*packed, sc)]
        for mode in ("batched", "plain"):
            b.align(sc, mode)
            got.append(b.results())
        b.close()
        for k, g in enumerate(got):
            for f in gbsw.FIELDS:
                assert np.array_equal(g[f], exp[f]), (k, f)
    finally:
        ctx.close()
