"""V(r) gathers the atoms near each brick of 8 x 8 x 4 points
(k_build_potential): the sum must stay that of every atom at every point, bit
for bit with linear tables, on grids that end inside a brick, with atoms
outside the box, tables of different ranges (one shorter than a grid spacing)
and atom counts around the 256 of one gathering round."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(24, 36, 16), (36, 24, 48), (80, 16, 24)])
@pytest.mark.parametrize("natom", [1, 256, 257, 600])
def test_bricks_vs_oracle(sep, oracle, grid, natom):
    print("case potential bricks", grid, natom, flush=True)
    rng = np.random.default_rng(natom)
    d = np.array([0.6, 0.75, 0.7])
    half = 0.5 * d * grid
    xyz = rng.uniform(-1.3, 1.3, (natom, 3)) * half
    types = rng.integers(0, 3, natom).astype(np.int32)
    npot = np.array([501, 301, 40])
    dr = np.array([0.01, 0.02, 0.01])
    vr = np.arange(501)[None, :] * dr[:, None]
    pot = -np.exp(-vr ** 2 / np.array([[2.0], [4.0], [0.05]])) + 0.01
    for t in range(3):
        pot[t] -= pot[t, npot[t] - 1]
    scale = rng.uniform(0.9, 1.1, natom)
    ref = oracle.build_potential(grid, tuple(-half), tuple(d), xyz, types, scale, npot, vr, pot,
                                 dr, (0.3, 5.0, 0.7))
    with sep.Context(*grid, *d, *-half) as ctx:
        got = ctx.build_potential(xyz, types, npot, vr, pot, dr, scale=scale, expot=(0.3, 5.0, 0.7))
        # the outer potential's exponential is the libraries' own on each side
        assert np.abs(got - ref).max() <= 1e-15 * np.abs(ref).max()
        assert ctx.vmin == got.min() and ctx.vmax == got.max()
        none = (0.0, 0.0, 1.0)
        ref = oracle.build_potential(grid, tuple(-half), tuple(d), xyz, types, scale, npot, vr,
                                     pot, dr, none)
        got = ctx.build_potential(xyz, types, npot, vr, pot, dr, scale=scale, expot=none)
        assert np.array_equal(got, ref)
