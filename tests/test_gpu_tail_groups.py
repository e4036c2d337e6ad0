"""The tail in groups of neighbouring smaller ids (k_tail_count, k_tail_split,
k_tail_group): candidates spread over the ids, heaped on some of them, on one
id beyond what a group holds, rounds and query sets. Every output is compared
whole with the oracle's and with the sorting passes' (a tuned tail keeps to
them)."""
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


def shuffled(seqs, seed):
    return [seqs[i] for i in np.random.default_rng(seed).permutation(len(seqs))]


def heaped(n, stars, rays, first):
    # `stars` strings of 16 residues with `rays` relatives one substitution away
    # (the star's own place among the ids is `first` of them or the last), among
    # n strings with no relatives
    rng = np.random.default_rng(stars + rays)
    rest = random_seqs(rng, n, 12, 16)
    centres = random_seqs(rng, stars, 16, 16)
    near = []
    for s in centres:
        k = 0
        while k < rays:
            i, c = k % 16, "ACDEFGHIKLMNPQRSTVWY"[k // 16]
            near.append(s[:i] + c + s[i + 1:])
            k += 1
    other = shuffled(rest + near, 5)
    return xtn.encode(centres + other if first else other + centres)


@pytest.mark.parametrize("name,make,d,measure", [
    ("spread", lambda: xtn.synth_nn(301, 30_000, planted=0.3, max_edits=1), 1, 0),
    ("spread", lambda: xtn.synth_nn(302, 200_000, planted=0.3, max_edits=1), 1, 1),
    ("spread", lambda: xtn.synth_nn(303, 131_073, planted=0.3, max_edits=2), 2, 0),
    ("spread", lambda: xtn.synth_nn(304, 700_000, planted=0.5, max_edits=2), 2, 0),
    ("spread", lambda: xtn.synth_nn(305, 12_000, planted=0.3, max_edits=3), 3, 1),
    ("spread", lambda: xtn.synth_nn(306, 900, planted=0.3, max_edits=3), 4, 0),
    ("spread", lambda: xtn.synth_nn(307, 120, planted=0.3, max_edits=3), 5, 0),
    ("few ids", lambda: xtn.encode(shuffled(random_seqs(np.random.default_rng(308), 300, 14, 14) * 7, 1)), 1, 0),
    ("heaped first", lambda: heaped(40_000, 20, 300, True), 1, 0),
    ("heaped last", lambda: heaped(40_000, 20, 300, False), 1, 0),
    # pairs among 320 relatives of one string: 50 000 candidates on 320 ids
    ("dense", lambda: heaped(30_000, 1, 320, True), 2, 0),
    # 260 equal rows and one more at the start, thirteen candidates a pair: the
    # first of them hold more than a group
    ("one id", lambda: xtn.encode(["CASSLGQETQYF"] + random_seqs(np.random.default_rng(309), 30_000, 14, 16)
                                  + ["CASSLGQETQYF"] * 260), 1, 0),
])
def test_grouped_tail_matches_oracle(name, make, d, measure):
    chars, offsets = make()
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, measure=measure) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for _ in range(3):  # eager, captured, replayed
            assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), want), eng.stats()
        eng.configure(max_pairs_per_round=20_000)
        assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), want)
        eng.configure(max_pairs_per_round=0)
        eng.set_tuning(sort_low_bits=8)
        assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), want)


def test_replays_of_other_rows_in_groups_and_passes():
    # the same counts and buffers: spread candidates, then thousands on one id
    rng = np.random.default_rng(310)
    base = random_seqs(rng, 40_000, 15, 15)
    spread = [s[:7] + "W" + s[8:] for s in base[:20_000]] + base[:20_000]
    star = "CASSLAPGATNEKLF"
    rays = [star[:i] + c + star[i + 1:] for i in range(15) for c in "ACDEFGHIKLMNPQRSTVWY"]
    rays += [r[:j] + c + r[j + 1:] for r in rays[:40] for j in range(15) for c in "ACDEFGHIKLMNPQRSTVWY"]
    heaps = (rays + base)[:40_000]
    inputs = [xtn.encode(shuffled(spread, 1)), xtn.encode(shuffled(heaps, 2))]
    want = [oracle.nn_port_mt(*x, 1, 0, THREADS)[0].astype(np.int64) for x in inputs]
    with xtn.Engine(distance=1) as eng:
        for _ in range(2):
            for x, w in zip(inputs, want):
                eng.set_sequences(chars=x[0], offsets=x[1])
                for _ in range(3):
                    assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), w)
