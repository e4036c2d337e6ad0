"""What a search learns about its rows (that they leave the tiles, need bins
in parts, or a tail in passes) holds for those rows at that distance, not for
other searches of the handle."""
import numpy as np
import pytest

import oracle
import xtn
from helpers import random_seqs

pytestmark = pytest.mark.gpu


def tiles(eng, search):
    eng.kernel_profile_reset()
    out = search()
    return out, eng.kernel_profile("tiles")[0]


def test_a_distance_out_of_the_tiles_leaves_the_others_in():
    # 1100 strings of four residues all share the empty variant at d = 4, more
    # records of one key than the bins' lists follow
    seqs = random_seqs(np.random.default_rng(420), 1100, 4, 4, unique=True)
    chars, offsets = xtn.encode(seqs)
    with xtn.Engine(distance=1, profile=True) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for d in (4, 1, 4, 2, 1):
            eng.configure(distance=d)
            (p, dist), tiled = tiles(eng, lambda: eng.copy_nn_output(eng.nn_resident()))
            want = oracle.nn_port_mt(chars, offsets, d, 0, 8)[0].astype(np.int64)
            assert np.array_equal(np.concatenate([p, dist.astype(np.int64)[:, None]], axis=1), want), d
            assert d == 4 or tiled == 1, d


def test_a_set_out_of_the_tiles_leaves_the_others_in():
    sets = [xtn.decode(*xtn.synth_nn(421 + k, 3_000, planted=0.3, max_edits=1)) for k in range(4)]
    sets[1] += ["CASSLGTDTQYF"] * 1100
    cuts = np.concatenate([[0], np.cumsum([len(s) for s in sets])]).astype(np.uint32)
    chars, offsets = xtn.encode([s for part in sets for s in part])
    with xtn.Engine(distance=1, profile=True) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        want = eng.nn_sets(cuts, batched=True)
        for first in (True, False):
            got, tiled = tiles(eng, lambda: eng.nn_sets(cuts, batched=False))
            assert got.keys() == want.keys()
            assert all(np.array_equal(got[k], want[k]) for k in want)
            assert tiled == (4 if first else 3)
