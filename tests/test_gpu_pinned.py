"""GPU test of uploads where pinned memory is not to be had: batches and calls of every
upload form are then copied from pageable memory, with the same results.  In a child
process, whose hipHostMalloc is a stand-in that refuses (host/pinned_shim.cpp)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

CHILD = r"""
import ctypes, os, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
import gbsw
from gbsw import synth

refuse_from = ctypes.c_long.in_dll(shim, "refuse_from")
refused = ctypes.c_long.in_dll(shim, "refused")
sc = gbsw.dna_scoring()
# one block, a scan on the device, and (above 8 MiB) the pinned ring
works = [synth.batched_dna(n, seed=0x5EED0710 + n) for n in (3, 1000, 20000)]
# all there; none at all; only small pieces (no ring)
contexts = [(gbsw.Context(0), 0), (gbsw.Context(0), 1), (gbsw.Context(0), 2 << 20)]
got = []
for ctx, limit in contexts:
    refuse_from.value, refused.value = limit, 0
    res = []
    for w in works:
        print("pinned memory refused from", limit, "bytes:", w.n, flush=True)
        args = (w.ref, w.ref_off, w.query, w.query_off)
        assert w.n < 20000 or len(w.ref) + len(w.query) > (8 << 20)
        res.append(ctx.align_packed(*args, sc))
        b = ctx.batch(gbsw.DNA, *args)
        b.align(sc)
        res.append(b.results())
        b.close()
    got.append(res)
    assert (refused.value > 0) == (limit > 0)
for x, y, z in zip(*got):
    for f in gbsw.FIELDS:
        assert np.array_equal(x[f], y[f]) and np.array_equal(x[f], z[f]), f
refuse_from.value = 0
w = works[2]
b = contexts[1][0].batch(gbsw.DNA, w.ref, w.ref_off, w.query, w.query_off) # and with it again
b.align(sc)
assert all(np.array_equal(b.results()[f], got[0][5][f]) for f in gbsw.FIELDS)
b.close()
for ctx, _ in contexts:
    ctx.close()
print("same results")
"""


def test_uploads_without_pinned_memory(tmp_path):
    shim = str(tmp_path / "pinned_shim.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", os.path.join(HERE, "host", "pinned_shim.cpp"), "-o", shim,
                    "-Wl,--no-as-needed", "-L" + os.path.join(ROCM, "lib"), "-lamdhip64",
                    "-Wl,-rpath," + os.path.join(ROCM, "lib"), "-ldl"], check=True)
    pkg = os.path.join(os.path.dirname(HERE), "gpu-bsw_amd")
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, shim, pkg], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip().endswith("same results"), r.stdout + r.stderr
