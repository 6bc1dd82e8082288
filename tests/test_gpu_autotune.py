"""GPU test: the autotuner times a plan once, however many geometry models make it.  A
batch of one short pair has one plan under every model, so that tuning it takes about as
long as the runs of one model (the six models' runs take six times as long)."""
import time

import numpy as np
import pytest

import gbsw

pytestmark = pytest.mark.gpu


def test_models_of_one_plan_are_timed_once():
    ctx = gbsw.Context(0)
    try:
        off = np.array([0, 20], dtype=np.uint64)
        seq = np.frombuffer(b"ACGTTGCAAGCTTACGGATC", dtype=np.uint8)
        sc = gbsw.dna_scoring()
        b = ctx.batch(gbsw.DNA, seq, off, seq, off)
        for _ in range(20):
            b.align(sc)
        repeats = 400
        t0 = time.perf_counter()
        for _ in range(repeats + 1):
            b.align(sc)
        once = time.perf_counter() - t0
        t0 = time.perf_counter()
        model, ms = b.autotune(sc, repeats)
        tuned = time.perf_counter() - t0
        assert 0 <= model < 6 and ms > 0
        assert tuned < 3 * once, "autotune %.4f s, %d runs %.4f s" % (tuned, repeats + 1, once)
        assert b.results()["score"][0] == 60
        b.close()
    finally:
        ctx.close()
