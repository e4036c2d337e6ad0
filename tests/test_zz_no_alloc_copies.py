"""The search without device allocation on rows that come several times: the
resident search's output, and the refusal of more candidates than the scratch
holds, at the counts where its route changes."""
import numpy as np
import pytest

import xtn
from test_zz_no_alloc import hip_runtime, noalloc, resident

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,copies,d,measure,status", [
    (1000, 6, 1, 0, 0), (2000, 4, 1, 1, 0), (340, 20, 1, 0, 6), (300, 15, 1, 0, 0), (200, 30, 1, 0, 6), (40, 200, 1, 0, 6),
    (300, 3, 2, 0, 0), (120, 5, 2, 1, 0), (400, 3, 2, 0, 0), (1000, 3, 2, 0, 0), (900, 4, 2, 0, 0), (1000, 6, 2, 0, 6),
    (100, 3, 3, 0, 0), (20, 3, 4, 0, 0),
])
def test_noalloc_copies(n, copies, d, measure, status):
    lib, hip = xtn.load_library(), hip_runtime()
    seqs = xtn.decode(*xtn.synth_nn(64, n, planted=0.3, max_edits=1)) * copies
    chars, offsets = xtn.encode([seqs[i] for i in np.random.default_rng(n).permutation(len(seqs))])
    for _ in range(2):
        st, got = noalloc(lib, hip, chars, offsets, d, measure, 1 << 20)
        assert st == status
        assert status or np.array_equal(got, resident(chars, offsets, d, measure))


@pytest.mark.parametrize("seed,n,copies,d,status", [(1, 230, 3, 3, 6), (2, 350, 10, 2, 6), (3, 54, 30, 2, 6),
                                                    (4, 18, 4, 4, 0), (5, 300, 3, 2, 0), (6, 40, 3, 3, 0),
                                                    (7, 2000, 2, 1, 0)])
def test_noalloc_strings_of_runs(seed, n, copies, d, status):
    # deleting any residue of a run gives the same string: many equal records
    # of one row, which count against the scratch's room
    rng = np.random.default_rng(seed)
    seqs = ["".join("ACDE"[int(rng.integers(0, 4))] * int(rng.integers(1, 4)) for _ in range(int(rng.integers(2, 8))))
            for _ in range(n)]
    chars, offsets = xtn.encode([s for s in seqs for _ in range(copies)])
    st, got = noalloc(xtn.load_library(), hip_runtime(), chars, offsets, d, 0, 1 << 20)
    assert st == status
    assert status or np.array_equal(got, resident(chars, offsets, d, 0))
