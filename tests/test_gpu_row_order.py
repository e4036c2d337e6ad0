"""Rows sorted by length, short and long ones standing together, on the GPU:
the same output as the oracle's, by the same kernels as shuffled rows."""
import os

import numpy as np
import pytest

import oracle
import xtn
from helpers import random_seqs

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def cdr3(seed, n, d, *lengths):
    return xtn.decode(*xtn.synth_nn(seed, n, *lengths, planted=0.3, max_edits=min(d, 2)))


def two_lengths(seed, n, short, long):
    # a quarter of short rows, a quarter a substitution away from long ones
    rng = np.random.default_rng(seed)
    seqs = random_seqs(rng, n // 4, short, short, unique=True) + random_seqs(rng, n // 2, long, long)
    return seqs + [s[:k % long] + "W" + s[k % long + 1:] for k, s in enumerate(seqs[-(n // 4):])]


@pytest.mark.parametrize("make,d,measure", [
    (lambda: two_lengths(301, 64_000, 5, 18), 1, 0),
    (lambda: cdr3(302, 99_991, 2, 15.0, 2.5, 6, 30), 2, 1),
    (lambda: cdr3(303, 40_000, 3), 3, 0),
    (lambda: two_lengths(304, 2_300, 8, 18), 4, 0),
])
@pytest.mark.parametrize("falling", [False, True])
def test_rows_sorted_by_length(make, d, measure, falling):
    chars, offsets = xtn.encode(sorted(make(), key=len, reverse=falling))
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, measure=measure) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for _ in range(3):  # eager, captured, replayed
            p, dist = eng.copy_nn_output(eng.nn_resident())
            assert np.array_equal(np.concatenate([p, dist.astype(np.int64)[:, None]], axis=1), want)
            assert eng.stats()["coarse_in_generator"] == 1


@pytest.mark.parametrize("falling", [False, True])
def test_overlap_of_rows_sorted_by_length(falling):
    # the lengths of the unique rows are counted on the device
    seqs = sorted(cdr3(305, 40_000, 1, 15.0, 2.5, 6, 30) + two_lengths(306, 20_000, 5, 18), key=len, reverse=falling)
    rng = np.random.default_rng(307)
    seqs = [s for s in seqs for _ in range(1 + len(s) % 2)]
    chars, offsets = xtn.encode(seqs)
    freq, rep = rng.integers(1, 50, len(seqs)), rng.integers(0, 6, len(seqs))
    want = oracle.overlap_mt(chars, offsets, freq, rep, 2, 0, THREADS)
    with xtn.Engine(distance=2) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for _ in range(2):
            assert np.array_equal(eng.overlap(freq, rep), want)
            assert eng.stats()["coarse_in_generator"] == 1
