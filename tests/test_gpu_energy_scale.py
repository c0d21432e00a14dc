"""The power iteration of the spectral bound (sep_energy_range) at units far
from 1: grid spacings scaled by 2^-k and V and Ekinmax by 2^2k scale H by 2^2k
exactly, the normalised start vector and every sum by powers of two, so that
the energies must be the unscaled ones times 2^2k to the last bit, after the
same number of iterations.  A steep V alone (1e20 Ha on an ordinary grid) is
checked against the oracle's iteration."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _range(sep, grid, d, V, k):
    s = 2.0 ** -k
    with sep.Context(*grid, d[0] * s, d[1] * s, d[2] * s, ekinmax=10.0 * 4.0 ** k) as ctx:
        ctx.set_potential(V * 4.0 ** k)
        return ctx.energy_range()


@pytest.mark.parametrize("grid", [(16, 16, 16), (24, 16, 32)])
def test_power_iteration_scales(sep, grid):
    V = np.random.default_rng(3).uniform(-1.5, 1.0, int(np.prod(grid)))
    d = (0.7, 0.8, 0.9)
    dE0, e0, it0 = _range(sep, grid, d, V, 0)
    assert np.isfinite(dE0) and it0 > 8
    for k in (-40, -32, 32, 36):
        dE, e, it = _range(sep, grid, d, V, k)
        print("case range", grid, "2^", 2 * k, dE, e, it, flush=True)
        assert it == it0
        assert e == e0 * 4.0 ** k and dE == dE0 * 4.0 ** k


@pytest.mark.parametrize("grid", [(16, 16, 16), (24, 16, 32)])
@pytest.mark.parametrize("scale", [1e20, 1e30])
def test_steep_potential(sep, oracle, grid, scale):
    V = np.random.default_rng(4).uniform(-1.5, 1.0, int(np.prod(grid))) * scale
    d = (0.7, 0.8, 0.9)
    ksq = oracle.ksqr(*grid, *d)
    dE_o, e_o, it_o = oracle.energy_range(grid, ksq, V, d[0] * d[1] * d[2], V.min())
    with sep.Context(*grid, *d) as ctx:
        ctx.set_potential(V)
        dE, e, it = ctx.energy_range()
    print("case steep", grid, scale, dE, e, it, "oracle", dE_o, e_o, it_o, flush=True)
    assert it == it_o
    # dE = 1.1 (e - vmin) cancels: held to the iteration's scale
    assert abs(e - e_o) <= 1e-10 * abs(e_o) and abs(dE - dE_o) <= 1e-10 * abs(e_o)
