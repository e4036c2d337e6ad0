"""Bins near and over the slots of the few-slot form, on the GPU: the search
stays in tiles."""
import os

import numpy as np
import pytest

import oracle
import xtn

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def search(eng, want):
    eng.kernel_profile_reset()
    p, dist = eng.copy_nn_output(eng.nn_resident())
    assert np.array_equal(np.concatenate([p, dist.astype(np.int64)[:, None]], axis=1), want)
    return {k: eng.kernel_profile(k)[0] for k in ("tiles", "gen", "gen_coarse")}


@pytest.mark.parametrize("seed,n", [(1, 178_000), (3, 178_000), (1, 176_000)])
def test_bins_near_their_slots(seed, n):
    # the means of these leave the 512 bins a few groups of room, which a bin
    # or two of the first two would outgrow
    chars, offsets = xtn.synth_nn(seed, n, planted=0.3, max_edits=1)
    want = oracle.nn_port_mt(chars, offsets, 1, 0, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=1, profile=True) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        assert search(eng, want) == dict(tiles=1, gen=0, gen_coarse=0)


def test_bin_over_its_slots():
    # 950 copies of one string over all tiles: its variants' bins outgrow the
    # form of few slots
    seqs = xtn.decode(*xtn.synth_nn(440, 165_000, planted=0.3, max_edits=1)) + ["CASLGTDTQYF"] * 950
    chars, offsets = xtn.encode([seqs[i] for i in np.random.default_rng(440).permutation(len(seqs))])
    want = oracle.nn_port_mt(chars, offsets, 1, 0, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=1, profile=True) as eng:
        for _ in range(2):  # what the first rows brought about ends with them
            eng.set_sequences(chars=chars, offsets=offsets)
            assert search(eng, want) == dict(tiles=2, gen=0, gen_coarse=0)
            assert search(eng, want) == dict(tiles=1, gen=0, gen_coarse=0)
