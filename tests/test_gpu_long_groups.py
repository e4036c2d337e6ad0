"""Many records of one key, on the GPU: pairs that outnumber the bins' list of
them, groups around the lengths that send a search to the bins in parts (64)
and out of the tiles (1024)."""
import os

import numpy as np
import pytest

import oracle
import xtn

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


@pytest.mark.parametrize("n,d,measure,copies", [
    # bins of few slots, whose list holds 1024 pairs
    (4_000, 1, 0, 45), (4_000, 1, 1, 47), (4_000, 2, 0, 65), (4_000, 1, 0, 1024), (4_000, 1, 0, 1025),
    # bins of 18 groups, with rounds (2400 pairs) and without
    (210_000, 1, 0, 64), (210_000, 1, 1, 65), (210_000, 1, 0, 66), (210_000, 1, 0, 600), (60_000, 2, 0, 70),
    (60_000, 2, 1, 200),
    # bins of 9 groups
    (12_000, 3, 0, 60), (2_600, 4, 0, 50),
])
def test_long_groups(n, d, measure, copies):
    seqs = xtn.decode(*xtn.synth_nn(450 + d, n, planted=0.3, max_edits=1)) + ["CASLGTDTQYF"] * copies
    chars, offsets = xtn.encode([seqs[i] for i in np.random.default_rng(copies).permutation(len(seqs))])
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, measure=measure) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for k in range(4):  # eager runs and replays; then in rounds of the smaller id
            eng.configure(profile=int(k == 3), max_pairs_per_round=1 << 17 if k == 3 and copies <= 1024 else 0)
            eng.kernel_profile_reset()
            p, dist = eng.copy_nn_output(eng.nn_resident())
            assert np.array_equal(np.concatenate([p, dist.astype(np.int64)[:, None]], axis=1), want), k
        assert eng.kernel_profile("tiles")[0] == (copies <= 1024)
