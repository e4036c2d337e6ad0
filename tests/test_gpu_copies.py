"""Rows that come several times, on the GPU: the records stay in tiles, with
the oracle's output, also where equal pairs outnumber the records; one string
of more copies than a bin's lists follow goes through the generator's coarse
pass, which writes no record for a repeated variant, and not through the
separate pass."""
import os

import numpy as np
import pytest

import oracle
import xtn

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def repeated(seed, n, copies):
    seqs = [s for s in xtn.decode(*xtn.synth_nn(seed, n, planted=0.3, max_edits=1)) for _ in range(copies)]
    return [seqs[i] for i in np.random.default_rng(seed).permutation(len(seqs))]


def launches(eng, *names):
    return {k: eng.kernel_profile(k)[0] for k in names}


def searched(eng, want):
    """a first search of new rows and a second one: the second's kernels"""
    for _ in range(2):
        eng.kernel_profile_reset()
        p, dist = eng.copy_nn_output(eng.nn_resident())
        assert np.array_equal(np.concatenate([p, dist.astype(np.int64)[:, None]], axis=1), want)
    return launches(eng, "tiles", "bins", "gen", "gen_coarse")


@pytest.mark.parametrize("n,copies,d,measure", [(6_000, 3, 2, 0), (30_000, 4, 1, 1), (2_000, 3, 3, 0), (900, 20, 2, 0),
                                                (400, 60, 1, 0), (300, 3, 4, 0)])
def test_copies_stay_in_tiles(n, copies, d, measure):
    chars, offsets = xtn.encode(repeated(400 + copies + d, n, copies))
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, measure=measure, profile=True) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        assert searched(eng, want) == dict(tiles=1, bins=1, gen=0, gen_coarse=0)


@pytest.mark.parametrize("n,d,measure", [(9_000, 2, 0), (60_000, 1, 1), (2_000, 3, 0)])
def test_outgrown_tiles_go_to_the_coarse_pass(n, d, measure):
    # one string 1100 times, spread over the rows
    seqs = xtn.decode(*xtn.synth_nn(410 + d, n, planted=0.3, max_edits=1)) + ["CASSLGTDTQYF"] * 1100
    chars, offsets = xtn.encode([seqs[i] for i in np.random.default_rng(d).permutation(len(seqs))])
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, measure=measure, profile=True) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        assert searched(eng, want) == dict(tiles=0, bins=0, gen=0, gen_coarse=1)
        assert d == 1 or eng.stats()["n_records"] < eng.stats()["n_variants"]
