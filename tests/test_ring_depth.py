"""Depth of the filter's ring of Newton vectors (csrc/sep_host.c): up to 1024
vectors in 32 GB, beyond that 256 or 32 a target, and whole sixteens where
memory is short, which the complex64 accumulation needs at its blocks' starts."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def host(sep):
    from semi_empirical_pseudopotentials_amd._lib import LIB_PATH
    L = ctypes.CDLL(LIB_PATH)
    L.sep_ring_depth.restype = ctypes.c_long
    L.sep_ring_depth.argtypes = [ctypes.c_long, ctypes.c_long, ctypes.c_double, ctypes.c_long]
    L.sep_ring_halve.restype = ctypes.c_long
    L.sep_ring_halve.argtypes = [ctypes.c_long]
    return L


def _per_k(n, ns, size):
    return float((ns + 1) // 2 * 2 * n ** 3 * size)


@pytest.mark.parametrize("nc,ms,per_k,most,want", [
    (4096, 32, _per_k(128, 16, 4), 1024, 1024),  # 137 GB for 32 targets
    (512, 1, _per_k(128, 8, 8), 1024, 256),      # 34 GB for one
    (4096, 1, _per_k(64, 8, 8), 1024, 1024),     # 17 GB
    (4096, 1, _per_k(80, 16, 8), 1024, 512),     # what fits 32 GB, in 64s
    (4096, 9, _per_k(160, 24, 4), 1024, 288),    # 32 a target
    (100, 40, _per_k(160, 24, 8), 1024, 100),
    (4096, 40, _per_k(160, 24, 8), 1024, 1024),
    (96, 4, _per_k(24, 3, 8), 32, 32),
    (1, 1, _per_k(16, 1, 4), 1024, 1),
])
def test_depth(host, nc, ms, per_k, most, want):
    assert host.sep_ring_depth(nc, ms, per_k, most) == want


@pytest.mark.parametrize("k", [1024, 960, 832, 576, 512, 352, 300, 288, 256, 100, 40, 33, 32, 17])
def test_halving_keeps_sixteens(host, k):
    while k > 8:
        h = host.sep_ring_halve(k)
        assert k // 2 - 16 < h <= k // 2
        assert h % 16 == 0 or h < 16
        k = h
