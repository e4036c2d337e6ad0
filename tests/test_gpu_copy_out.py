"""xtn_copy_nn_output into pageable and pinned memory, whole and in part, below
and above the size of the readback's staging, at odd addresses."""
import ctypes

import numpy as np
import pytest
import torch

import xtn

pytestmark = pytest.mark.gpu


def room(kind, nbytes, skew):
    if kind == "pinned":
        return torch.full((nbytes + 64,), 7, dtype=torch.uint8, pin_memory=True).numpy()[skew:skew + nbytes]
    return np.full(nbytes + 64, 7, dtype=np.uint8)[skew:skew + nbytes]


@pytest.fixture(scope="module")
def searched():
    chars, offsets = xtn.synth_nn(460, 600_000, planted=0.4, max_edits=1)
    with xtn.Engine(distance=1) as eng:
        eng.set_sequences(chars=chars, offsets=offsets)
        n = eng.nn_resident()
        pairs, dist = eng.copy_nn_output(n)
        yield eng, pairs, dist


@pytest.mark.parametrize("kinds", [("pageable", "pageable"), ("pinned", "pinned"), ("pinned", "pageable"),
                                   ("pageable", "pinned")])
@pytest.mark.parametrize("share", [0.001, 0.3, 1.0, 1.5])
def test_output_into_any_host_memory(searched, kinds, share):
    eng, pairs, dist = searched
    assert 9 * len(dist) > 2 << 20
    cap = int(share * len(dist))
    n = min(cap, len(dist))
    p, d = room(kinds[0], 8 * cap, 8), room(kinds[1], cap, 3)
    assert eng.lib.xtn_copy_nn_output(eng.h, ctypes.cast(p.ctypes.data, ctypes.POINTER(xtn.Int2)),
                                      ctypes.cast(d.ctypes.data, ctypes.POINTER(ctypes.c_int8)), cap) == 0
    assert np.array_equal(p[:8 * n].view(np.int32).reshape(-1, 2), pairs[:n]) and (p[8 * n:] == 7).all()
    assert np.array_equal(d[:n].view(np.int8), dist[:n]) and (d[n:] == 7).all()
