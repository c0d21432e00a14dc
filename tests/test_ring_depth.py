"""Depth of the filter's ring of Newton vectors (csrc/sep_host.c): up to 1024
vectors in 32 GB, beyond that 256 or 32 a target, and whole sixteens where
memory is short, which the complex64 accumulation needs at its blocks' starts.
Grids of a batch share the memory without taking from one another what the
others do not use."""
import ctypes

import numpy as np
import pytest


@pytest.fixture(scope="module")
def host(sep):
    from semi_empirical_pseudopotentials_amd._lib import LIB_PATH
    L = ctypes.CDLL(LIB_PATH)
    L.sep_ring_plan.restype = None
    L.sep_ring_halve.restype = ctypes.c_long
    L.sep_ring_halve.argtypes = [ctypes.c_long]
    return L


def _plan(host, grids, total, most=1024):
    """Depths of (nc, ms, per_k) grids."""
    nc, ms = (np.array([g[i] for g in grids], dtype=np.int64) for i in (0, 1))
    per_k = np.array([g[2] for g in grids])
    K = np.zeros(len(grids), dtype=np.int64)
    p = [a.ctypes.data_as(ctypes.c_void_p) for a in (nc, ms, per_k)]
    host.sep_ring_plan(len(grids), *p, ctypes.c_long(most), ctypes.c_double(total),
                       K.ctypes.data_as(ctypes.c_void_p))
    return [int(k) for k in K]


def _per_k(n, ns, size):
    return float((ns + 1) // 2 * 2 * n ** 3 * size)


@pytest.mark.parametrize("nc,ms,per_k,most,want", [
    (4096, 32, _per_k(128, 16, 4), 1024, 1024),  # 137 GB for 32 targets
    (512, 1, _per_k(128, 8, 8), 1024, 256),      # 34 GB for one
    (4096, 1, _per_k(64, 8, 8), 1024, 1024),     # 17 GB
    (4096, 1, _per_k(80, 16, 8), 1024, 512),     # what fits 32 GB, in 64s
    (4096, 9, _per_k(160, 24, 4), 1024, 288),    # 32 a target
    (4096, 9, _per_k(160, 36, 4), 1024, 144),    # 288 would take 170 GB
    (100, 40, _per_k(160, 24, 8), 1024, 100),
    (4096, 40, _per_k(160, 24, 8), 1024, 128),   # 805 GB
    (96, 4, _per_k(24, 3, 8), 32, 32),
    (1, 1, _per_k(16, 1, 4), 1024, 1),
])
def test_depth(host, nc, ms, per_k, most, want):
    assert _plan(host, [(nc, ms, per_k)], 160e9, most) == [want]


@pytest.mark.parametrize("k", [1024, 960, 832, 576, 512, 352, 300, 288, 256, 100, 40, 33, 32, 17])
def test_halving_keeps_sixteens(host, k):
    while k > 8:
        h = host.sep_ring_halve(k)
        assert k // 2 - 16 < h <= k // 2
        assert h % 16 == 0 or h < 16
        k = h


def test_batch_of_unlike_grids(host):
    """Two 160^3 grids of one target (256 each, 67 GB) beside six small ones
    (1024 each, 18 GB in all) fit 100 GB as they are."""
    grids = [(2048, 1, _per_k(160, 8, 4))] * 2 + [(2048, 1, _per_k(48, 8, 4))] * 6
    assert _plan(host, grids, 100e9) == [256] * 2 + [1024] * 6
    # 75 GB: the small ones come down to what the large ones want; 50 GB: all do
    assert _plan(host, grids, 75e9) == [256] * 8
    assert _plan(host, grids, 50e9) == [128] * 8


@pytest.mark.parametrize("total", [1e6, 1e9, 20e9, 170e9, 1e12])
def test_plan_fits_or_is_least(host, total):
    rng = np.random.default_rng(6)
    for _ in range(200):
        grids = [(int(rng.integers(1, 5000)), int(rng.integers(1, 50)),
                  _per_k(int(rng.choice([16, 36, 64, 128, 160])), int(rng.integers(1, 40)),
                         int(rng.choice([4, 8])))) for _ in range(rng.integers(1, 9))]
        alone = [_plan(host, [g], 1e30)[0] for g in grids]
        K = _plan(host, grids, total)
        assert all(1 <= k <= a for k, a in zip(K, alone))
        assert sum(k * g[2] for k, g in zip(K, grids)) <= total or max(K) <= 8
        assert all(k == a or k == max(K) for k, a in zip(K, alone))
