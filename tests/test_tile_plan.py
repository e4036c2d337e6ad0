"""The plan of tiles and bins (xtn_plan.hpp) on the CPU, over lengths in any
order: no tile gets more sequences than its tables and indexes take, nor more
records than its slots."""
import ctypes
import math
import os
import subprocess

import numpy as np
import pytest

from conftest import PKG

SOURCE = """
#include "xtn_plan.hpp"
extern "C" void plan(const int64_t* counts, int64_t n, int d, int n_cu, int64_t* out) {
	xtn::LenCounts len;
	for (int L = 0; L <= xtn::MAX_PREFIX; ++L)
		len.c[L] = counts[L];
	const xtn::TilePlan p = xtn::plan_tiles(len, n, d, n_cu);
	const int64_t v[] = {p.tile, p.least, p.ntiles, p.slot_bits, p.bin_bits, p.idx_bits, p.bin_nt, p.bin_groups};
	for (int k = 0; k < 8; ++k)
		out[k] = v[k];
}
extern "C" int seqs(int d) { return xtn::tl_seqs(d); }
"""
FIELDS = ("tile", "least", "ntiles", "slot_bits", "bin_bits", "idx_bits", "bin_nt", "bin_groups")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-shared", "-fPIC", "-I", os.path.join(PKG, "csrc"), "-o",
                    str(d / "plan.so"), str(d / "plan.cpp")], check=True, timeout=120)
    lib = ctypes.CDLL(str(d / "plan.so"))
    lib.plan.argtypes = [ctypes.c_void_p, ctypes.c_int64, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    return lib


def plan(lib, counts, d, n_cu=256):
    counts = np.ascontiguousarray(counts, dtype=np.int64)
    out = np.zeros(8, dtype=np.int64)
    lib.plan(counts.ctypes.data, int(counts.sum()), d, n_cu, out.ctypes.data)
    return dict(zip(FIELDS, out.tolist()))


def variants(d):
    return np.array([sum(math.comb(L, k) for k in range(min(d, L) + 1)) for L in range(19)], dtype=np.int64)


def lengths(name, n, rng):
    if name == "cdr3":
        return np.clip(np.rint(rng.normal(15, 2, n)), 8, 18).astype(np.int64)
    if name == "wide":
        return np.clip(np.rint(rng.normal(15, 2.5, n)), 6, 18).astype(np.int64)
    if name == "two":
        return np.where(rng.random(n) < 0.5, 4, 18)
    if name == "mostly long":
        return np.where(rng.random(n) < 0.02, 1, 18)
    if name == "short":
        return rng.integers(1, 6, n)
    return rng.integers(0, 19, n)  # any


@pytest.mark.parametrize("d,length,n", [(2, 1, 80_000_000), (1, 2, 100_000_000), (2, 2, 60_000_000), (4, 1, 30_000_000),
                                        (1, 18, 20_000_000), (2, 18, 2_500_000), (3, 18, 400_000), (4, 18, 100_000)])
def test_tiles_and_slots_have_room_for_their_numbers(lib, d, length, n):
    # a listed record keeps its tile in 16 bits, a group of records its first
    # slot in 30
    counts = np.zeros(19, dtype=np.int64)
    counts[length] = n
    p = plan(lib, counts, d)
    assert p["ntiles"] <= 65535
    assert p["ntiles"] << p["slot_bits"] < 1 << 30


@pytest.mark.parametrize("d", [1, 2, 3, 4])
@pytest.mark.parametrize("name", ["cdr3", "wide", "two", "mostly long", "short", "any"])
@pytest.mark.parametrize("n", [37, 3_001, 60_013, 700_001])
def test_tiles_hold_lengths_in_any_order(lib, d, name, n):
    rng = np.random.default_rng(n + d)
    L = lengths(name, n, rng)
    v = variants(d)
    p = plan(lib, np.bincount(L, minlength=19), d)
    if p["ntiles"] == 0:  # more records than the bins take
        assert v[L].sum() > 3e8
        return
    limit = min(lib.seqs(d), (1 << p["idx_bits"]) - 1)
    assert p["slot_bits"] <= 15
    for order in (L, np.sort(L), np.sort(L)[::-1], np.concatenate([np.sort(L[::2]), np.sort(L[1::2])])):
        w = np.maximum(v[order], p["least"])
        tile = (np.cumsum(w) - w) // p["tile"]
        assert p["ntiles"] == -(-int(w.sum()) // p["tile"]) > tile[-1]
        assert np.bincount(tile).max() <= limit
        assert np.bincount(tile, weights=v[order]).max() <= 1 << p["slot_bits"]
