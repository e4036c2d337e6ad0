"""The searches a program runs through this package, as measured cases.

Every case goes through the package's public entry points (xtn.Engine,
xtn.Server, xtn_nn_noalloc) on seeded synthetic CDR3 sets of the generator
that the tests and bench.py use: unique strings of about 15 residues, a share
of them planted within a few edits of an earlier one. A pass ends with the
whole output in the caller's hands: the sorted (i, j, distance) triples, the
repertoire matrix, or the answers of every query. The caller's buffers hold
more triples than any input of the case gives; the count comes back with them.

`exact` has nothing to add: every output is a whole number (row indexes,
distances, frequency sums), which has to be equal.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xt-neighbor_amd"))

import xtn  # noqa: E402

LENGTHS = {  # mean, deviation, shortest, longest
    "cdr3": (15.0, 2.0, 8, 22),
    "wide": (15.0, 2.5, 6, 30),  # the lengths of the 5M-sequence workload
}
MEASURES = {"leven": xtn.LEVENSHTEIN, "hamming": xtn.HAMMING}


def listed():
    return [
        # a search inside a program that may not allocate: one small repertoire on the device, latency only
        dict(name="noalloc-1k-d1", kind="noalloc", n=1009, distance=1, measure="leven", lengths="cdr3"),
        # the command line's smallest everyday input, host strings in and triples out
        dict(name="nn-10k-d1-host", kind="nn", n=10_000, distance=1, measure="leven", lengths="cdr3", upload=True),
        # one ordinary repertoire, same-length neighbours, searched again on a handle that holds it
        dict(name="nn-100k-hamming-d2", kind="nn", n=99_991, distance=2, measure="hamming", lengths="wide", upload=False),
        # a wider search of one repertoire (the distance sweep's third point)
        dict(name="nn-100k-d3", kind="nn", n=100_000, distance=3, measure="leven", lengths="cdr3", upload=False),
        # the distance sweep's fourth point, on half the rows: deletion sets beyond three positions
        dict(name="nn-50k-d4", kind="nn", n=50_000, distance=4, measure="leven", lengths="cdr3", upload=False),
        # the whole drop-in boundary at an ordinary size: check, upload, search, triples in host memory
        dict(name="nn-300k-d2-host", kind="nn", n=300_007, distance=2, measure="leven", lengths="cdr3", upload=True),
        # the headline workload: a million sequences at distance 2
        dict(name="nn-1M-d2", kind="nn", n=1_000_000, distance=2, measure="leven", lengths="cdr3", upload=False),
        # many sequences at distance 1 (a cohort's pooled repertoires)
        dict(name="nn-5M-d1", kind="nn", n=5_000_000, distance=1, measure="leven", lengths="wide", upload=False),
        # the largest: 3.7e8 deletion variants, more than one key-space chunk holds
        dict(name="nn-3M-d2", kind="nn", n=3_000_000, distance=2, measure="leven", lengths="cdr3", upload=False),
        # overlap of two dozen repertoires (duplicates across them, frequencies in, matrix out)
        dict(name="overlap-24", kind="overlap", n=24, distance=1, measure="leven", size_min=10_000, size_max=60_000),
        # many query sets in one call
        dict(name="sets-400-d2", kind="sets", n=400_000, distance=2, measure="leven", lengths="cdr3", sets=400),
        # query sets against a resident index
        dict(name="served-2M-d1", kind="served", n=2_000_000, distance=1, measure="leven", lengths="cdr3", queries=16,
             query_min=1000, query_max=50_000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# rows at each distance that generate about 3.5e8 variants, at most
MOST_ROWS = {1: 5_000_000, 2: 2_800_000, 3: 400_000, 4: 60_000}


def draw(rng):
    kind = rng.choice(["nn", "nn", "nn", "nn", "noalloc", "overlap", "sets", "served"])
    measure = rng.choice(["leven", "leven", "hamming"])
    lengths = rng.choice(["cdr3", "wide"])
    if kind == "noalloc":
        d = rng.choice([1, 2])
        return dict(kind=kind, n=_log_int(rng, 200, 40_000 if d == 1 else 6000), distance=d, measure=measure,
                    lengths=lengths)
    if kind == "overlap":
        return dict(kind=kind, n=rng.randint(2, 40), distance=rng.choice([1, 1, 2]), measure=measure,
                    size_min=_log_int(rng, 500, 5000), size_max=_log_int(rng, 6000, 40_000))
    if kind == "sets":
        n = _log_int(rng, 5000, 1_000_000)
        return dict(kind=kind, n=n, distance=rng.choice([1, 2]), measure=measure, lengths=lengths,
                    sets=rng.randint(2, max(2, n // 500)))
    if kind == "served":
        return dict(kind=kind, n=_log_int(rng, 50_000, 2_000_000), distance=1, measure=measure, lengths=lengths,
                    queries=rng.randint(1, 24), query_min=500, query_max=_log_int(rng, 1000, 50_000))
    d = rng.choice([1, 1, 2, 2, 2, 3, 4])
    return dict(kind=kind, n=_log_int(rng, 1000, MOST_ROWS[d]), distance=d, measure=measure, lengths=lengths,
                upload=rng.choice([True, False]))


class Held:
    """what a program holds between calls, released with it"""

    def __init__(self, case, **parts):
        self.case = case
        self.__dict__.update(parts)

    def __del__(self):
        for owner in ("engine", "server"):
            if owner in self.__dict__:
                self.__dict__[owner].close()


def _strings(case, seed, n):
    mu, sigma, lmin, lmax = LENGTHS[case["lengths"]]
    return xtn.synth_nn(seed + 1, n, mu, sigma, lmin, lmax, planted=0.25, max_edits=min(case["distance"], 2))


def _room(case, n):
    """output triples the caller makes room for (about 0.3 a row come at distances 1 and 2)"""
    return (1 if case["distance"] <= 2 else 4) * n + 4096


def _keep(out, at, pairs, dist):
    """one answer into the caller's buffers"""
    out["pairs"][at:at + len(pairs)] = pairs
    out["dist"][at:at + len(dist)] = dist
    return at + len(pairs)


def _query_sizes(case):
    return [int(s) for s in np.geomspace(case["query_min"], case["query_max"], case["queries"])]


def prepare(case, seed):
    kind, d, measure = case["kind"], case["distance"], MEASURES[case["measure"]]
    if kind == "overlap":
        chars, offsets, freq, sizes = xtn.synth_overlap(seed + 1, case["n"], case["size_min"], case["size_max"],
                                                        shared=0.1)
        engine = xtn.Engine(distance=d, measure=measure)
        engine.set_sequences(chars=chars, offsets=offsets)
        return Held(case, engine=engine, freq=freq, rep=xtn.reps_from_sizes(sizes),
                    matrix=np.zeros((case["n"] * (case["n"] + 1) // 2, 3), np.int64))
    chars, offsets = _strings(case, seed, case["n"])
    if kind == "noalloc":
        room = _room(case, case["n"])
        return Held(case, lib=xtn.load_library(),
                    chars=torch.from_numpy(np.concatenate([chars, np.zeros(16, np.uint8)])).cuda(),
                    offsets=torch.from_numpy(offsets.astype(np.int32)).cuda(),
                    out={"pairs": torch.zeros((room, 2), dtype=torch.int32, device="cuda"),
                         "dist": torch.zeros(room, dtype=torch.int8, device="cuda")})
    rows = sum(_query_sizes(case)) if kind == "served" else case["n"]
    room = _room(case, rows)
    out = {"pairs": np.zeros((room, 2), np.int32), "dist": np.zeros(room, np.int8)}
    if kind == "served":
        queries = [xtn.synth_queries(seed * 1000 + k + 1, chars, offsets, s, planted=0.3)
                   for k, s in enumerate(_query_sizes(case))]
        server = xtn.Server(chars, offsets, distance=d, measure=measure, slots=4, max_query_rows=1 << 17)
        return Held(case, server=server, queries=queries, out=out)
    engine = xtn.Engine(distance=d, measure=measure)
    if kind == "sets":
        engine.set_sequences(chars=chars, offsets=offsets)
        rng = np.random.default_rng(seed)
        cuts = np.concatenate([[0], np.cumsum(np.exp(rng.uniform(math.log(100), math.log(10_000), case["sets"])))])
        return Held(case, engine=engine, out=out, cuts=np.round(cuts / cuts[-1] * case["n"]).astype(np.uint32))
    if not case["upload"]:
        engine.set_sequences(chars=chars, offsets=offsets)
    return Held(case, engine=engine, chars=chars, offsets=offsets, out=out)


def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "overlap":
        rows = state.engine.overlap(state.freq, state.rep)
        state.matrix[:len(rows)] = rows
        return {"matrix": state.matrix, "count": len(rows)}
    out = state.out
    if kind == "nn" and case["upload"]:
        state.engine.set_sequences(chars=state.chars, offsets=state.offsets)
        pairs, dist, _ = state.engine.nn()
        return {**out, "count": _keep(out, 0, pairs, dist)}
    if kind == "nn":
        engine = state.engine
        count = engine.nn_resident()
        status = engine.lib.xtn_copy_nn_output(engine.h, out["pairs"].ctypes.data_as(ctypes.POINTER(xtn.Int2)),
                                               out["dist"].ctypes.data_as(ctypes.POINTER(ctypes.c_int8)),
                                               len(out["dist"]))
        if status != 0 or count > len(out["dist"]):
            raise RuntimeError(f"xtn_copy_nn_output: status {status}, {count} pairs")
        return {**out, "count": count}
    if kind == "noalloc":
        count = ctypes.c_int64()
        status = state.lib.xtn_nn_noalloc(state.chars.data_ptr(), state.offsets.data_ptr(), case["n"],
                                          case["distance"], MEASURES[case["measure"]], out["pairs"].data_ptr(),
                                          out["dist"].data_ptr(), out["dist"].numel(), ctypes.byref(count), None)
        if status != 0:
            raise RuntimeError(f"xtn_nn_noalloc: status {status}")
        return {**out, "count": count.value}
    if kind == "sets":
        counts, at = np.zeros(case["sets"], np.int64), 0
        for k, triples in state.engine.nn_sets(state.cuts).items():
            counts[k] = len(triples)
            at = _keep(out, at, triples[:, :2], triples[:, 2])
        return {**out, "counts": counts}
    tickets = [state.server.submit(*q) for q in state.queries]
    counts, at = np.zeros(len(tickets), np.int64), 0
    for k, t in enumerate(tickets):
        pairs, dist, _ = state.server.wait(t)
        counts[k] = len(pairs)
        at = _keep(out, at, pairs, dist)
    return {**out, "counts": counts}


def _mean_variants(lengths, d):
    """deletion variants of a sequence: the sum over at most d deletions of its 18-residue prefix"""
    mu, sigma, lmin, lmax = LENGTHS[lengths]
    weight = {L: math.exp(-0.5 * ((L - mu) / sigma) ** 2) for L in range(lmin, lmax + 1)}
    total = sum(weight.values())
    return sum(w / total * sum(math.comb(min(L, 18), k) for k in range(min(d, L) + 1)) for L, w in weight.items())


def work(case):
    """Bytes: every string and offset in once, every triple out once (about one
    planted pair for four rows). Operations: each deletion variant named by one
    multiply-add per deletion, each pair's band of the distance table filled once."""
    d = case["distance"]
    if case["kind"] == "overlap":
        n = int(case["n"] * (case["size_max"] - case["size_min"]) / math.log(case["size_max"] / case["size_min"]))
        lengths = "cdr3"
    elif case["kind"] == "served":  # the index is resident: the query rows
        n, lengths = sum(_query_sizes(case)), case["lengths"]
    else:
        n, lengths = case["n"], case["lengths"]
    pairs = 0.25 * n
    return {"bytes": n * (15.0 + 4.0) + 9.0 * pairs,
            "flops": 2.0 * d * n * _mean_variants(lengths, d) + pairs * 15 * (2 * d + 1) * 4}


def exact(case, seed):
    return None
