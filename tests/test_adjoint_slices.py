"""How many slices the Hellmann-Feynman adjoint cuts an atom's box into
(hf_slices, csrc/sep_adjoint.hip): enough for a few atoms to fill the GPU, and no
more reductions of partial sums than they are worth for many."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def slices(sep):
    from semi_empirical_pseudopotentials_amd._lib import LIB_PATH
    fn = getattr(ctypes.CDLL(LIB_PATH), "_ZN3sep9hf_slicesEldi")  # sep::hf_slices(long, double, int)
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_long, ctypes.c_double, ctypes.c_int]
    return fn


# atoms, points of a box, pairs of a pass, (least, most) slices whose calls lie
# within 6 % of the fastest measured
@pytest.mark.parametrize("natom,box,pairs,least,most", [
    (1, 13824.0, 1, 10, 64), (1, 29791.0, 1, 4, 64), (10, 13824.0, 4, 3, 24),
    (10, 29791.0, 8, 8, 32), (100, 13824.0, 1, 2, 8), (100, 13824.0, 8, 2, 5),
    (100, 29791.0, 1, 3, 20), (100, 29791.0, 8, 2, 5), (300, 13824.0, 8, 1, 1),
    (300, 29791.0, 4, 1, 5), (693, 29791.0, 1, 1, 6), (693, 29791.0, 8, 1, 2),
    (1000, 29791.0, 1, 1, 3)])
def test_measured_ranges(slices, natom, box, pairs, least, most):
    assert least <= slices(natom, box, pairs) <= most


@pytest.mark.parametrize("natom", [1, 2, 511, 512, 513, 100000, 30000000])
@pytest.mark.parametrize("box", [1.0, 64.0, 4.1e6])
@pytest.mark.parametrize("pairs", [1, 2, 4, 8])
def test_bounds(slices, natom, box, pairs):
    n = slices(natom, box, pairs)
    assert 1 <= n <= 64 and natom * n < 2 ** 31
