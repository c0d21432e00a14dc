"""V(r) of a geometry with one NaN coordinate: every point NaN and the extrema at
their start values (filter/init.c:116-117), whichever coordinate it is, so that a
relaxation that has run away is seen; an atom at infinity adds nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interp", [0, 1])
@pytest.mark.parametrize("grid", [(24, 24, 24), (16, 36, 24)])
def test_nan_and_infinite_atoms(sep, grid, interp):
    rng = np.random.default_rng(8)
    d = 0.8
    half = [-n * d / 2 for n in grid]
    npot, dr = np.array([200, 150]), np.array([0.02, 0.02])
    vr = np.arange(200)[None] * dr[:, None]
    pot = rng.uniform(-1, 1, (2, 200))
    xyz = rng.uniform(-6, 6, (300, 3))
    types = rng.integers(0, 2, 300).astype(np.int32)
    with sep.Context(*grid, d, d, d, *half) as ctx:
        ctx.set_interp(interp)

        def V(x):
            return ctx.build_potential(x, types, npot, vr, pot, dr)

        print("case potential nan", grid, interp, flush=True)
        assert np.isfinite(V(xyz)).all()
        for atom in (0, 255, 256, 299):
            for k in range(3):
                bad = xyz.copy()
                bad[atom, k] = np.nan
                assert np.isnan(V(bad)).all(), (atom, k)
                assert ctx.vmin == 1.0e10 and ctx.vmax == -1.0e10
        far = xyz.copy()
        far[17] = [np.inf, -np.inf, 0.0]
        without = ctx.build_potential(np.delete(xyz, 17, 0), np.delete(types, 17), npot, vr, pot, dr)
        assert np.array_equal(V(far), without)
