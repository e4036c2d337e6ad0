"""The tiled record path (xtn_tiles.hpp) on the GPU, where it can go wrong:
the smallest inputs that take it, a last tile of a few records, string lengths
around the 18-residue prefix and very short ones (tiles of more sequences than
their tables hold, which go to the separate pass), rows repeated so often that
a bin lists more records than fit (bins in parts), query sets, and rounds of
the smaller id. Every output is compared whole with the oracle's."""
import os

import numpy as np
import pytest

import oracle
import xtn
from helpers import random_seqs

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def triples(p, d):
    return np.concatenate([p.astype(np.int64), d.astype(np.int64)[:, None]], axis=1)


def search(eng, d, measure, **cfg):
    eng.configure(distance=d, measure=measure, **cfg)
    return triples(*eng.copy_nn_output(eng.nn_resident())), eng.stats()


def repeated(seed, n, copies, **kw):
    seqs = xtn.decode(*xtn.synth_nn(seed, n, planted=0.3, max_edits=1, **kw))
    seqs = [s for s in seqs for _ in range(copies)]
    order = np.random.default_rng(seed).permutation(len(seqs))
    return xtn.encode([seqs[i] for i in order])


def mixed_lengths(seed, n):
    # a quarter each of 2 to 5, 6 to 12, 17 to 19 and 24 to 40 residues, relatives among the long ones
    rng = np.random.default_rng(seed)
    long = random_seqs(rng, n // 8, 24, 40)
    near = [s[:20] + "A" + s[21:] if k % 2 else s[:3] + s[4:] for k, s in enumerate(long)]
    seqs = random_seqs(rng, n // 4, 2, 5) + random_seqs(rng, n // 4, 6, 12) + random_seqs(rng, n // 4, 17, 19)
    seqs += long + near
    return xtn.encode([seqs[i] for i in rng.permutation(len(seqs))])


@pytest.mark.parametrize("name,make,d,measure,tiled", [
    # about 600 000 variants, the fewest that are tiled, and a few more
    ("smallest", lambda: xtn.synth_nn(101, 38_000, planted=0.3, max_edits=1), 1, 0, None),
    ("smallest", lambda: xtn.synth_nn(102, 5_000, planted=0.3, max_edits=2), 2, 1, None),
    ("smallest", lambda: xtn.synth_nn(103, 1_100, planted=0.3, max_edits=2), 3, 0, None),
    ("ragged", lambda: xtn.synth_nn(104, 70_001, 15.0, 2.5, 6, 30, planted=0.3, max_edits=2), 2, 0, 1),
    ("ragged", lambda: xtn.synth_nn(105, 25_013, 15.0, 2.5, 6, 30, planted=0.3, max_edits=3), 3, 1, 1),
    ("smallest", lambda: xtn.synth_nn(116, 320, planted=0.4, max_edits=2), 4, 0, None),
    ("ragged", lambda: xtn.synth_nn(117, 6_007, 15.0, 2.5, 6, 30, planted=0.3, max_edits=3), 4, 0, 1),
    ("mixed lengths", lambda: mixed_lengths(118, 2_400), 4, 1, None),
    ("mixed lengths", lambda: mixed_lengths(106, 24_000), 2, 0, None),
    ("mixed lengths", lambda: mixed_lengths(107, 6_000), 3, 0, None),
    ("all one length", lambda: xtn.synth_nn(108, 60_000, 18.0, 0.0, 18, 18, planted=0.3, max_edits=1), 1, 0, 1),
    ("short strings", lambda: xtn.synth_nn(109, 40_000, 7.0, 0.0, 7, 7, planted=0.2, max_edits=1), 2, 0, None),
    # every record has one copy: the bins' lists run over and the bins go in parts
    ("twice", lambda: repeated(113, 30_000, 2), 2, 0, 1),
    ("twice", lambda: repeated(114, 90_000, 2), 1, 0, 1),
    ("twice", lambda: repeated(115, 7_000, 2), 3, 1, 1),
    # more equal pairs than records: the separate pass
    ("copies", lambda: repeated(110, 20_000, 3), 2, 0, 0),
    ("copies", lambda: repeated(111, 60_000, 4), 1, 1, 0),
    ("copies", lambda: repeated(112, 5_000, 3), 3, 0, 0),
])
def test_tiled_search_matches_oracle(name, make, d, measure, tiled):
    chars, offsets = make()
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for _ in range(3):  # eager, captured, replayed
            got, st = search(eng, d, measure)
            assert np.array_equal(got, want), (name, st)
        assert tiled is None or st["coarse_in_generator"] == tiled
        # the separate pass and back
        got, _ = search(eng, d, measure, coarse_separate=1)
        assert np.array_equal(got, want)
        got, _ = search(eng, d, measure, coarse_separate=0)
        assert np.array_equal(got, want)


def fifteens(seed, n):
    # 15 residues each, a third of the rows a substitution away from another
    seqs = random_seqs(np.random.default_rng(seed), n - n // 3, 15, 15)
    return xtn.encode(seqs + [s[:k % 15] + "W" + s[k % 15 + 1:] for k, s in enumerate(seqs[:n // 3])])


@pytest.mark.parametrize("name,make,d,measure,tiled", [
    # 16 variants each: 4080, 4096 and 4112 records around the fewest that are tiled
    ("fewest", lambda: fifteens(201, 255), 1, 0, 0),
    ("fewest", lambda: fifteens(202, 256), 1, 1, 1),
    ("fewest", lambda: fifteens(203, 257), 1, 0, 1),
    ("fewest", lambda: xtn.synth_nn(204, 41, planted=0.3, max_edits=2), 2, 0, None),
    ("fewest", lambda: xtn.synth_nn(205, 9, planted=0.3, max_edits=2), 3, 0, None),
    ("fewest", lambda: xtn.synth_nn(206, 3, planted=0.3, max_edits=2), 4, 1, None),
    # bins in number up to two per CU, then the forms of more slots
    ("more bins", lambda: xtn.synth_nn(207, 17_001, planted=0.3, max_edits=1), 1, 0, 1),
    ("more bins", lambda: xtn.synth_nn(208, 2_003, 15.0, 2.5, 6, 30, planted=0.3, max_edits=2), 2, 0, 1),
    ("few slots", lambda: xtn.synth_nn(209, 19_009, planted=0.3, max_edits=2), 2, 1, 1),
    ("few slots", lambda: xtn.synth_nn(210, 2_311, planted=0.3, max_edits=2), 3, 0, 1),
    ("few slots", lambda: xtn.synth_nn(211, 1_000, planted=0.3, max_edits=2), 4, 0, 1),
    ("mixed lengths", lambda: mixed_lengths(212, 400), 3, 1, None),
    ("mixed lengths", lambda: mixed_lengths(213, 4_000), 1, 0, None),
    ("short strings", lambda: xtn.synth_nn(214, 3_000, 6.0, 0.0, 6, 6, planted=0.2, max_edits=1), 2, 0, None),
    ("twice", lambda: repeated(215, 700, 2), 2, 0, None),
    ("copies", lambda: repeated(216, 40, 60), 1, 0, 0),
    ("one row", lambda: xtn.encode(["CASSLGTDTQYF"] * 500), 1, 0, 0),
])
def test_tiled_small_inputs(name, make, d, measure, tiled):
    test_tiled_search_matches_oracle(name, make, d, measure, tiled)


@pytest.mark.parametrize("d", [1, 2, 3])
def test_tiled_sets_and_rounds(d):
    n = {1: 60_000, 2: 30_000, 3: 8_000}[d]
    chars, offsets = xtn.synth_nn(120 + d, n, planted=0.4, max_edits=d)
    want = oracle.nn_port_mt(chars, offsets, d, 0, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        got, st = search(eng, d, 0, max_pairs_per_round=4096)
        assert np.array_equal(got, want)
        assert st["n_rounds"] > 1 and st["coarse_in_generator"] == 1
        eng.configure(max_pairs_per_round=0)
        cuts = np.array([0, 7, 7, n // 3, n - 1, n], dtype=np.uint32)
        for _ in range(3):
            got = eng.nn_sets(cuts)
            for k in range(len(cuts) - 1):
                a, b = int(cuts[k]), int(cuts[k + 1])
                inside = want[(want[:, 0] >= a) & (want[:, 1] < b)] - np.array([a, a, 0])
                assert np.array_equal(got.get(k, np.zeros((0, 3), np.int64)), inside), k


def test_replays_keep_their_distance():
    # a captured run of one distance, runs of others, and the captured one again
    # (few candidates at every distance, so that the plan for them stays)
    long = random_seqs(np.random.default_rng(130), 7_000, 13, 17)
    chars, offsets = xtn.encode(long + [s[:k] + "AC"[k % 2] + s[k + k % 3:] for k, s in enumerate(long[:8])])
    want = {d: oracle.nn_port_mt(chars, offsets, d, 0, THREADS)[0].astype(np.int64) for d in (2, 3, 4)}
    back = 0  # replays right after another distance's run
    with xtn.Engine(distance=2) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for d in (4, 3, 2):  # every buffer is there from here on: graphs stay valid
            assert np.array_equal(search(eng, d, 0)[0], want[d])
        for first, other in [(2, 3), (3, 2), (3, 4), (4, 2)]:
            for k, d in enumerate((first, first, first, other, first, first)):
                got, st = search(eng, d, 0)
                assert np.array_equal(got, want[d]), (first, other, d, st)
                back += st["graph_replays"] if k == 4 else 0
    assert back >= 1


@pytest.mark.parametrize("d,n", [(1, 120_000), (2, 24_000), (3, 8_000)])
def test_replays_with_other_rows_of_the_same_shape(d, n):
    # the same counts and buffers, so the same graph: rows all apart, then rows
    # of which each has one copy (the bins' lists run over) or many (more equal
    # pairs than records)
    def rows(copies):
        base = random_seqs(np.random.default_rng(140 + copies), n // copies, 15, 15)
        seqs = [s for s in base for _ in range(copies)]
        return xtn.encode([seqs[i] for i in np.random.default_rng(copies).permutation(n)])

    inputs = {c: rows(c) for c in (1, 2, 8)}
    want = {c: oracle.nn_port_mt(*inputs[c], d, 0, THREADS)[0].astype(np.int64) for c in inputs}
    with xtn.Engine(distance=d) as eng:
        eng.set_sequences(chars=inputs[1][0], offsets=inputs[1][1])
        for _ in range(3):
            got, st = search(eng, d, 0)
            assert np.array_equal(got, want[1])
        assert st["graph_replays"] == 1
        for c in (2, 1, 8, 2, 1):
            eng.set_sequences(chars=inputs[c][0], offsets=inputs[c][1])
            for _ in range(2):
                got, st = search(eng, d, 0)
                assert np.array_equal(got, want[c]), (c, st)
