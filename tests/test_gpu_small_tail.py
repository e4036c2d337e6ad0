"""The one-workgroup tail (k_tail_small): exact candidate counts around the
edges of its rows, its waves and its capacity, every distance's band, and the
served form. Every output is compared whole with the oracle's and with the
sorting passes' (a tuned tail keeps to them)."""
import os

import numpy as np
import pytest

import oracle
import xtn
from helpers import clustered_seqs, random_seqs

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def triples(p, d):
    return np.concatenate([p.astype(np.int64), d.astype(np.int64)[:, None]], axis=1)


def near_pairs(p):
    # p pairs one substitution apart, at a residue unlike its neighbours, which
    # share one variant at distance 1, met once; strings of 11 random residues
    # meet by chance about once in 600 inputs
    rng = np.random.default_rng(150 + p)
    left = random_seqs(rng, p + 2, 11, 11)
    right = []
    for s in left[:p]:
        k = int(rng.choice([i for i in range(11) if s[i] not in s[max(0, i - 1):i] + s[i + 1:i + 2]]))
        right.append(s[:k] + next(c for c in "ACDEFG" if c not in s[max(0, k - 1):k + 2]) + s[k + 1:])
    seqs = left + right
    return xtn.encode([seqs[i] for i in rng.permutation(len(seqs))])


@pytest.mark.parametrize("p", [0, 1, 63, 64, 65, 1023, 1024, 1025, 6000, 6001, 7169, 8191, 8192, 8193, 8250])
def test_candidate_counts(p):
    chars, offsets = near_pairs(p)
    want = oracle.nn_port_mt(chars, offsets, 1, 0, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=1) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for _ in range(3):  # the count unknown, then known; captured and replayed where it stays
            assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), want)
            assert eng.stats()["n_candidates"] == p
        eng.set_tuning(sort_low_bits=8)
        assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), want)


@pytest.mark.parametrize("measure", [0, 1])
@pytest.mark.parametrize("d,n,lmax", [(1, 3000, 26), (2, 700, 26), (3, 150, 26), (4, 60, 20), (5, 40, 16), (6, 40, 14),
                                      (7, 40, 12), (8, 40, 11), (9, 40, 11)])
def test_distances(d, n, lmax, measure):
    seqs = clustered_seqs(np.random.default_rng(160 + d), n, 1, lmax, edits=min(d, 3))
    chars, offsets = xtn.encode(seqs)
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, measure=measure) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for _ in range(3):
            assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), want)
        eng.set_tuning(sort_low_bits=8)
        assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), want)


def test_replay_with_more_candidates_than_it_takes():
    # the same counts of rows and residues, few candidates and then many
    few = near_pairs(4000)
    base = random_seqs(np.random.default_rng(170), 800, 11, 11)
    many = xtn.encode((base * 11)[:len(few[1]) - 1])
    want = [oracle.nn_port_mt(*x, 1, 0, THREADS)[0].astype(np.int64) for x in (few, many)]
    with xtn.Engine(distance=1) as eng:
        for _ in range(2):
            for x, w in zip((few, many), want):
                eng.set_sequences(chars=x[0], offsets=x[1])
                for _ in range(3):
                    assert np.array_equal(triples(*eng.copy_nn_output(eng.nn_resident())), w)


def test_served_queries_on_both_sides():
    rng = np.random.default_rng(180)
    rows = random_seqs(rng, 3000, 11, 15)
    ichars, ioffs = xtn.encode(rows + rows[:40] * 12)
    with xtn.Server(ichars, ioffs, distance=1, slots=2) as srv:
        for qs in (rows[100:400], rows[:40] * 8, rows[:3], rows[:40] * 9 + rows[50:900], rows[2000:2100]):
            qchars, qoffs = xtn.encode(qs)
            ni = len(ioffs) - 1
            tri, _ = oracle.nn_port(np.concatenate([ichars, qchars]),
                                    np.concatenate([ioffs, qoffs[1:] + ioffs[-1]]).astype(np.uint32), 1, 0)
            cross = tri[(tri[:, 0] < ni) & (tri[:, 1] >= ni)]
            want = np.stack([cross[:, 1] - ni, cross[:, 0], cross[:, 2]], axis=1).astype(np.int64)
            want = want[np.lexsort((want[:, 1], want[:, 0]))]
            p, dist, _ = srv.wait(srv.submit(qchars, qoffs))
            assert np.array_equal(triples(p, dist), want)
