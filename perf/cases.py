"""Performance cases of the alignment engine: what its users have it do, through its
public Python entry points.

A case is a plain dict.  `kind` names the entry point:

  align    one call on host buffers (Context.align_packed, or kernel_driver_aa on
           Python strings): packing or upload, both passes, results back on the host
  batch    one align of a batch that is resident on the GPU; the results stay there
           (gbsw_batch_device_results, read in place)
  paths    alignment paths (CIGAR words) of a resident, aligned batch
  serve    a burst of requests through the serving loop, until all are answered

Sequences: every query is a stretch of its own reference with substitutions and
single-residue indels (reads against contigs, homologous proteins), the model of
this repository's synthetic workloads.  Lengths are lognormal around `*_med` with
sigma 0.5, clipped to [lo, hi], or uniform in [lo, hi] where `*_med` is 0; with
`q_frac` the query takes a uniform 0.5 to 1.0 of its reference instead.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-bsw_amd"))

import gbsw  # noqa: E402
from gbsw.scoring import AA_ORDER, BLOSUM62  # noqa: E402
from gbsw.synth import AA_BACKGROUND  # noqa: E402

DNA_SCORES = (3, -3, -6, -1)
AA_GAPS = (-6, -1)
OPS_PER_CELL = 12  # integer operations of one affine-gap cell, as bench.py counts them

READS = dict(alphabet="dna", r_med=600, r_lo=64, r_hi=2048, q_med=150, q_lo=32, q_hi=1024, q_frac=False)
SHORT_READS = dict(alphabet="dna", r_med=0, r_lo=200, r_hi=1000, q_med=0, q_lo=100, q_hi=150, q_frac=False)
LONG_READS = dict(alphabet="dna", r_med=6000, r_lo=1500, r_hi=24000, q_med=4000, q_lo=1000, q_hi=16000, q_frac=False)
PROTEINS = dict(alphabet="protein", r_med=350, r_lo=50, r_hi=1024, q_med=0, q_lo=0, q_hi=0, q_frac=True)
LONG_PROTEINS = dict(alphabet="protein", r_med=0, r_lo=4096, r_hi=16384, q_med=0, q_lo=1024, q_hi=4096, q_frac=False)


def listed():
    return [
        # one read against one contig, the smallest call: its latency
        dict(name="one_read", kind="align", pairs=1, n_rate=0.0, strings=False, **READS),
        # what one thread of an assembler hands over at a time; some reads hold N
        dict(name="reads_300_call", kind="align", pairs=300, n_rate=0.001, strings=False, **READS),
        # a query's database hits as Python strings, through the reference's own entry point
        dict(name="proteins_200_strings", kind="align", pairs=200, n_rate=0.0, strings=True, **PROTEINS),
        # the whole way of an ordinary batch: upload, alignment, results; reads hold N
        dict(name="reads_150k_call", kind="align", pairs=150_000, n_rate=0.0005, strings=False, **READS),
        # short reads against contigs: the plain DNA benchmark set
        dict(name="short_reads_10k", kind="batch", pairs=10_000, n_rate=0.0, **SHORT_READS),
        # the headline benchmark: a million reads of uneven length
        dict(name="reads_1m", kind="batch", pairs=1_000_000, n_rate=0.0, **READS),
        # the plain protein benchmark set
        dict(name="proteins_20k", kind="batch", pairs=20_000, n_rate=0.0, **PROTEINS),
        # long proteins: the benchmark's distribution, a fifth of its pairs
        dict(name="long_proteins_10k", kind="batch", pairs=10_000, n_rate=0.0, **LONG_PROTEINS),
        # long reads against long contigs: few pairs, each far wider than a wavefront
        dict(name="long_reads_400", kind="batch", pairs=400, n_rate=0.0, **LONG_READS),
        # CIGARs of a batch of reads, and of a batch of proteins
        dict(name="reads_300k_paths", kind="paths", pairs=300_000, n_rate=0.0, **READS),
        dict(name="proteins_5k_paths", kind="paths", pairs=5_000, n_rate=0.0, **PROTEINS),
        # a burst on the serving loop: 96 requests of 1 to 4,096 pairs, 70 % reads, 30 % proteins
        dict(name="serve_96", kind="serve", requests=96, max_pairs=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: any entry point, sizes over their logarithm."""
    which = rng.choice(["call", "call", "reads", "reads", "proteins", "long", "paths", "serve"])
    rate = rng.choice([0.0, 0.0, 0.001])

    def lengths(base):
        d = dict(base)
        if d["r_med"]:
            d["r_med"] = max(d["r_lo"], int(d["r_med"] * rng.uniform(0.5, 1.3)))
        if d["q_med"]:
            d["q_med"] = max(d["q_lo"], int(d["q_med"] * rng.uniform(0.5, 1.3)))
        elif not d["q_frac"]:
            d["q_lo"] = rng.randint(max(1, d["q_lo"] // 2), d["q_lo"])
        return d

    if which == "call":
        base = rng.choice([READS, SHORT_READS, PROTEINS])
        n = _log_int(rng, 1, 100_000 if base["alphabet"] == "dna" else 10_000)
        aa = base["alphabet"] == "protein"
        return dict(kind="align", pairs=n, n_rate=0.0 if aa else rate, strings=aa and n < 2000, **lengths(base))
    if which == "reads":
        return dict(kind="batch", pairs=_log_int(rng, 500, 700_000), n_rate=rate,
                    **lengths(rng.choice([READS, SHORT_READS])))
    if which == "proteins":
        return dict(kind="batch", pairs=_log_int(rng, 200, 100_000), n_rate=0.0, **lengths(PROTEINS))
    if which == "long":
        base, most = rng.choice([(LONG_PROTEINS, 6000), (LONG_READS, 300)])
        return dict(kind="batch", pairs=_log_int(rng, 20, most), n_rate=0.0, **lengths(base))
    if which == "paths":
        base, most = rng.choice([(READS, 200_000), (SHORT_READS, 200_000), (PROTEINS, 5000)])
        return dict(kind="paths", pairs=_log_int(rng, 50, most), n_rate=0.0, **lengths(base))
    return dict(kind="serve", requests=rng.randint(8, 96), max_pairs=_log_int(rng, 64, 4096))


# ---------------------------------------------------------------- inputs

def _lengths(case, n, rng):
    def some(med, lo, hi):
        if med:
            return np.clip(np.rint(rng.lognormal(math.log(med), 0.5, n)), lo, hi).astype(np.int64)
        return rng.integers(lo, hi + 1, n)
    r = some(case["r_med"], case["r_lo"], case["r_hi"])
    if case["q_frac"]:
        q = np.maximum(1, np.rint(r * rng.uniform(0.5, 1.0, n))).astype(np.int64)
    else:
        q = some(case["q_med"], case["q_lo"], case["q_hi"])
        r = np.maximum(r, q)
    return r, np.minimum(q, r)


def _offsets(lens):
    off = np.zeros(len(lens) + 1, dtype=np.uint64)
    np.cumsum(lens, out=off[1:])
    return off


def _substitutions():
    """Row a: cumulative probability of the residue that replaces residue a."""
    p = np.array(AA_BACKGROUND)[None, :] * 2.0 ** (np.array(BLOSUM62).reshape(24, 24)[:20, :20] / 2.0)
    np.fill_diagonal(p, 0.0)
    return np.cumsum(p / p.sum(1, keepdims=True), 1)


def _sequences(case, n, seed):
    """(ref bytes, ref offsets, query bytes, query offsets) in host memory, made on the GPU."""
    dev = "cuda"
    gen = torch.Generator(dev).manual_seed(seed)
    rlen, qlen = _lengths(case, n, np.random.default_rng(seed))
    protein = case["alphabet"] == "protein"
    letters = AA_ORDER[:20] if protein else "ACGT"
    sub, indel = (0.30, 0.03) if protein else (0.10, 0.02)

    def uniform(k):
        return torch.rand(k, generator=gen, device=dev)

    cum_bg = torch.tensor(np.cumsum(AA_BACKGROUND), dtype=torch.float32, device=dev)

    def background(k):
        if protein:
            return torch.bucketize(uniform(k), cum_bg, right=True).clamp_(max=19).to(torch.uint8)
        return torch.randint(0, 4, (k,), generator=gen, device=dev, dtype=torch.uint8)

    ro = _offsets(rlen)
    ref = background(int(ro[-1]))
    lens = torch.from_numpy(qlen).to(dev)
    start = torch.from_numpy(ro[:-1].astype(np.int64) + (np.random.default_rng(seed + 1).random(n) *
                                                         (rlen - qlen + 1)).astype(np.int64)).to(dev)
    q_first = torch.cumsum(lens, 0) - lens
    total = int(qlen.sum())
    src = torch.repeat_interleave(start - q_first, lens, output_size=total) + torch.arange(total, device=dev)
    q = ref[src]
    del src
    hit = uniform(total) < sub
    old = q[hit]
    if protein:
        cum = torch.tensor(_substitutions(), dtype=torch.float32, device=dev)
        u = uniform(len(old))
        q[hit] = (cum[old.long()] <= u[:, None]).sum(1).clamp_(max=19).to(torch.uint8)
    else:
        q[hit] = (old + torch.randint(1, 4, (len(old),), generator=gen, device=dev, dtype=torch.uint8)) % 4
    u = uniform(total)
    dele, ins = u < indel / 2, (u >= indel / 2) & (u < indel)
    dele[q_first] = False  # no query loses all its residues
    reps = 1 - dele.long() + ins.long()
    at = torch.cumsum(reps, 0)
    kept = torch.zeros(n + 1, dtype=torch.long, device=dev)
    kept[1:] = at[q_first + lens - 1]
    q = torch.repeat_interleave(q, reps, output_size=int(at[-1]))
    slots = at[ins] - 1
    q[slots] = background(len(slots))
    table = torch.tensor(list(letters.encode()), dtype=torch.uint8, device=dev)

    def text(codes):
        out = table[codes.int()]
        if case["n_rate"] > 0:
            out[uniform(len(out)) < case["n_rate"]] = ord("N")
        return out.cpu().numpy()

    return text(ref), ro, text(q), kept.cpu().numpy().astype(np.uint64)


def _scoring(case):
    if case["alphabet"] == "dna":
        return gbsw.dna_scoring(*DNA_SCORES)
    return gbsw.protein_scoring(BLOSUM62, *AA_GAPS)


class _DeviceArray:
    """int32 device memory of a batch's results, for torch.as_tensor.  It holds the
    batch, which owns the memory: a tensor made of it may outlive the state."""

    def __init__(self, batch, ptr, shape):
        self.batch = batch
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<i4", "version": 2}


def _device_results(batch):
    p = ctypes.c_void_p()
    if gbsw.load_library().gbsw_batch_device_results(batch._h, ctypes.byref(p)) != 0:
        raise RuntimeError("gbsw_batch_device_results failed")
    return torch.as_tensor(_DeviceArray(batch, p.value, (5, batch.n)), device="cuda")


def _requests(case):
    """The burst's requests; their sizes are the case's, their sequences the seed's."""
    rng = np.random.default_rng(case["requests"])
    sizes = np.exp(rng.uniform(0.0, math.log(case["max_pairs"]), case["requests"])).astype(int)
    protein = rng.random(case["requests"]) >= 0.7
    return [(dict(READS, n_rate=0.0) if not p else dict(PROTEINS, n_rate=0.0), int(s)) for s, p in zip(sizes, protein)]


def prepare(case, seed):
    if case["kind"] == "serve":
        reqs = [(c, _sequences(c, n, seed + 7 * k)) for k, (c, n) in enumerate(_requests(case))]
        buf = gbsw.HostBuffer(sum(len(s[0]) + len(s[2]) for _, s in reqs) + 16)  # pinned: read in place
        results = np.zeros(sum(5 * (len(s[1]) - 1) for _, s in reqs), dtype=np.int32)
        at, to, out = 0, 0, []
        for c, (r, ro, q, qo) in reqs:
            n, pairs = len(r) + len(q), len(ro) - 1
            buf.array[at:at + len(r)] = r
            buf.array[at + len(r):at + n] = q
            out.append((_scoring(c), ro + np.uint64(at), qo + np.uint64(at + len(r)),
                        results[to:to + 5 * pairs].reshape(5, pairs)))
            at += n
            to += 5 * pairs
        return dict(kind="serve", server=gbsw.Server(0), buf=buf, requests=out, results=results)
    r, ro, q, qo = _sequences(case, case["pairs"], seed)
    sc = _scoring(case)
    if case["kind"] == "align":
        state = dict(kind="align", seqs=(r, ro, q, qo), scoring=sc, strings=case["strings"])
        if case["strings"]:
            rt, qt = r.tobytes().decode(), q.tobytes().decode()
            state["contigs"] = [rt[int(a):int(b)] for a, b in zip(ro[:-1], ro[1:])]
            state["reads"] = [qt[int(a):int(b)] for a, b in zip(qo[:-1], qo[1:])]
        return state
    batch = gbsw.default_context().batch(sc.alphabet, r, ro, q, qo)
    state = dict(kind=case["kind"], batch=batch, scoring=sc)
    if case["kind"] == "batch":
        state["out"] = _device_results(batch)
        return state
    batch.align(sc)
    n = case["pairs"]
    state["words"] = np.zeros(n * (24 if case["alphabet"] == "dna" else 96) + 4096, dtype=np.uint32)
    state["offsets"] = np.zeros(n + 1, dtype=np.int64)
    state["path_score"] = np.zeros(n, dtype=np.int32)
    return state


def run(state):
    kind = state["kind"]
    if kind == "batch":
        state["batch"].align(state["scoring"])
        return tuple(state["out"])
    if kind == "paths":
        # the C entry point itself, into the caller's own buffers
        w, off, score = state["words"], state["offsets"], state["path_score"]
        if gbsw.load_library().gbsw_batch_traceback(state["batch"]._h, ctypes.byref(state["scoring"]), len(w),
                                                    w.ctypes.data, off.ctypes.data, score.ctypes.data, None) != 0:
            raise RuntimeError("gbsw_batch_traceback failed")
        return w.view(np.int32), off, score
    if kind == "serve":
        srv, a = state["server"], state["buf"].array
        sent = [srv.submit(sc, a, ro, a, qo, out)[0] for sc, ro, qo, out in state["requests"]]
        for ticket in sent:
            if srv.wait(ticket)["status"] != 0:
                raise RuntimeError("a request failed")
        return state["results"]
    if state["strings"]:
        res = gbsw.kernel_driver_aa(state["reads"], state["contigs"], BLOSUM62, *AA_GAPS)
    else:
        res = gbsw.default_context().align_packed(*state["seqs"], state["scoring"])
    return tuple(res[f] for f in gbsw.FIELDS)


# ---------------------------------------------------------------- what a pass cannot do without

def _pair_work(case, n):
    """(cells, residues) of n pairs, from a sample of the case's lengths."""
    r, q = _lengths(case, min(n, 50_000) if n > 2000 else 2000, np.random.default_rng(12345))
    return n * float(np.mean(r * q)), n * float(np.mean(r + q))


def work(case):
    if case["kind"] == "serve":
        parts = [_pair_work(c, n) + (n,) for c, n in _requests(case)]
        cells, residues, n = (sum(p[k] for p in parts) for k in range(3))
    else:
        n = case["pairs"]
        cells, residues = _pair_work(case, n)
    if case["kind"] == "paths":
        # the rectangles of the best alignments: about query length squared
        r, q = _lengths(case, min(n, 50_000), np.random.default_rng(12345))
        cells = n * float(np.mean(q.astype(np.float64) ** 2))
        return {"bytes": residues + n * (20 + 8 + 4 + 4 * 8), "flops": OPS_PER_CELL * cells}
    return {"bytes": residues + n * (16 + 20), "flops": OPS_PER_CELL * cells}


# ---------------------------------------------------------------- scores in 64 bits

def _scores(r, ro, q, qo, case):
    """Best local score of every pair, row by row over the references, 64-bit."""
    dev = "cuda"
    n = len(ro) - 1
    rl, ql = np.diff(ro).astype(np.int64), np.diff(qo).astype(np.int64)
    rows, cols = int(rl.max()), int(ql.max())

    def padded(buf, off, lens, width):
        first = torch.from_numpy(off[:-1].astype(np.int64)).to(dev)[:, None]
        j = torch.arange(width, device=dev)[None, :]
        inside = j < torch.from_numpy(lens).to(dev)[:, None]
        t = torch.from_numpy(np.ascontiguousarray(buf)).to(dev).long()
        return torch.where(inside, t[(first + j).clamp_(max=len(buf) - 1)], -1)

    a, b = padded(r, ro, rl, rows), padded(q, qo, ql, cols)
    if case["alphabet"] == "dna":
        match, mismatch, go, ge = DNA_SCORES
    else:
        go, ge = AA_GAPS
        code = torch.zeros(256, dtype=torch.long, device=dev)
        for k, c in enumerate(AA_ORDER):
            code[ord(c)] = k
        table = torch.tensor(list(BLOSUM62), dtype=torch.long, device=dev)
        ca, cb = code[a.clamp(min=0)], code[b.clamp(min=0)]
    low = -(1 << 40)
    h = torch.zeros(n, cols + 1, dtype=torch.long, device=dev)
    f = torch.full_like(h, low)
    best = torch.zeros(n, dtype=torch.long, device=dev)
    ramp = ge * torch.arange(cols + 1, device=dev)
    for i in range(rows):
        if case["alphabet"] == "dna":
            s = torch.where(a[:, i:i + 1] == b, match, mismatch)
        else:
            s = table[ca[:, i:i + 1] * 24 + cb]
        s = torch.where((b < 0) | (a[:, i:i + 1] < 0), low, s)
        f = torch.maximum(f + ge, h + go)
        top = torch.zeros_like(h)
        top[:, 1:] = h[:, :-1] + s
        top = torch.maximum(top, f).clamp_(min=0)
        # a gap along the row: the best earlier cell, open once, extend by distance
        gap = torch.cummax(top - ramp, 1).values[:, :-1] + ramp[1:] + go - ge
        h = top
        h[:, 1:] = torch.maximum(top[:, 1:], gap)
        inside = a[:, i:i + 1] >= 0
        best = torch.maximum(best, torch.where(inside & (b >= 0), h[:, 1:], 0).amax(1))
    return best.cpu().numpy()


def exact(case, seed):
    """The scores; where a best alignment begins and ends (and which of equal paths is
    taken) is the engine's own tie rule, a whole number with no 64-bit counterpart."""
    if case["kind"] not in ("align", "batch"):
        return None
    n = case["pairs"]
    r_most, q_most = case["r_hi"], case["q_hi"] or case["r_hi"]
    if n * r_most * q_most > 3e10:
        return None
    r, ro, q, qo = _sequences(case, n, seed)
    return (_scores(r, ro, q, qo, case), None, None, None, None)
