"""The generator's coarse pass of a single chunk, on the GPU: taken by
distances above 4 and by searches whose caller sets the chunk size, here at
least all records. The kernels that ran are asserted beside the oracle's
output: the pass, a sub-range that overflows, a region that overflows and is
regrouped from the compacted sub-ranges, and small buckets."""
import os

import numpy as np
import pytest

import oracle
import xtn
from test_gpu_coarse import runs_input

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)
KERNELS = ("tiles", "gen", "gen_coarse", "region", "sort_rec_scatter")


def search(eng, **cfg):
    eng.configure(**cfg)
    eng.kernel_profile_reset()
    p, dist = eng.copy_nn_output(eng.nn_resident())
    return np.concatenate([p, dist.astype(np.int64)[:, None]], axis=1), {k: eng.kernel_profile(k)[0] for k in KERNELS}


def shuffled(seed, n, share, copies):
    chars, offsets = xtn.synth_nn(seed, n, 14.0, 4.0, 4, 30, planted=0.3, max_edits=2)
    seqs = xtn.decode(chars, offsets)
    rng = np.random.default_rng(seed)
    seqs += [seqs[i] for i in rng.integers(0, n, int(share * n)) for _ in range(copies)]
    return xtn.encode([seqs[i] for i in rng.permutation(len(seqs))])


CASES = [
    ("ordinary", lambda: xtn.synth_nn(431, 45_000, planted=0.3, max_edits=1), 1, 0),
    ("ordinary", lambda: xtn.synth_nn(432, 20_000, planted=0.3, max_edits=2), 2, 1),
    ("uneven", lambda: shuffled(433, 70_000, 0.2, 3), 1, 1),
    ("uneven", lambda: shuffled(434, 30_000, 0.3, 2), 2, 0),
    ("uneven", lambda: shuffled(435, 9_000, 0.1, 2), 3, 0),
    ("runs", lambda: runs_input(2, 0), 2, 0),
    ("ordinary", lambda: xtn.synth_nn(436, 600, planted=0.3, max_edits=2), 5, 0),
]


@pytest.mark.parametrize("name,make,d,measure", CASES)
def test_coarse_pass_matches_oracle(name, make, d, measure):
    chars, offsets = make()
    want = oracle.nn_port_mt(chars, offsets, d, measure, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, measure=measure, profile=True, max_records_per_chunk=1 << 30) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for _ in range(2):
            got, ran = search(eng)
            assert np.array_equal(got, want), name
            st = eng.stats()
            assert ran["gen_coarse"] == 1 and ran["region"] == 1 and ran["tiles"] == ran["gen"] == 0
            assert st["coarse_in_generator"] == 1 and st["n_chunks"] == 1
            assert 0 < st["n_records"] <= st["n_variants"] - (d in (2, 3))


def test_sub_range_overflow_goes_to_the_separate_pass():
    # 455 copies of one string stand together: each of its 9 variants brings
    # 455 records to a sub-range of about 165 slots
    base = xtn.decode(*xtn.synth_nn(437, 45_000, planted=0.3, max_edits=1))
    chars, offsets = xtn.encode(["CDEFGHIK"] * 455 + base)
    want = oracle.nn_port_mt(chars, offsets, 1, 0, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=1, profile=True, max_records_per_chunk=1 << 30) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        for k in range(2):
            got, ran = search(eng)
            assert np.array_equal(got, want)
            assert ran["gen_coarse"] == (1 if k == 0 else 0) and ran["gen"] == 1 and ran["tiles"] == 0
            assert eng.stats()["coarse_in_generator"] == 0


@pytest.mark.parametrize("d,n,cap", [(2, 60_000, 75), (2, 60_000, 1650), (1, 45_000, 900)])
def test_region_overflow_is_regrouped(d, n, cap):
    chars, offsets = xtn.synth_nn(438, n, planted=0.3, max_edits=2)
    want = oracle.nn_port_mt(chars, offsets, d, 0, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=d, profile=True, max_records_per_chunk=1 << 30, bucket_capacity=cap) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        got, ran = search(eng)
        assert np.array_equal(got, want)
        assert ran["gen_coarse"] == 1 and ran["region"] == 1 and ran["tiles"] == ran["gen"] == 0
        assert ran["sort_rec_scatter"] > 0  # the exact sort of the compacted records


@pytest.mark.parametrize("cap,target,nt,tile", [(2048, 1500, 256, 4096), (4096, 3400, 512, 8192), (2048, 1230, 1024, 8192)])
def test_bucket_settings_of_the_coarse_pass(cap, target, nt, tile):
    chars, offsets = runs_input(3, 0)
    want = oracle.nn_port_mt(chars, offsets, 3, 0, THREADS)[0].astype(np.int64)
    with xtn.Engine(distance=3, profile=True, max_records_per_chunk=1 << 30) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        eng.set_tuning(bucket_capacity=cap, bucket_target=target, sort_threads=nt, sort_tile=tile)
        got, ran = search(eng)
        assert np.array_equal(got, want)
        assert ran["gen_coarse"] >= 1 and ran["tiles"] == 0
