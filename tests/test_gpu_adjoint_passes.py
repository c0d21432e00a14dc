"""The Hellmann-Feynman adjoint at every width of a pass: 1, 2, 4 or 8
densities at once, by their number (with a ragged last pass) and by the table
length whose histogram must fit in LDS; atoms of three types in mixed order,
one type without atoms, one atom alone.  FP64 sums of a few thousand points in
another order than the oracle's: 1e-11 of the largest value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,npairs,natom", [
    (401, 1, 1), (401, 2, 7), (401, 3, 40), (401, 9, 40),  # by the pairs: 1, 2, 4, 8 and 1
    (2433, 8, 5), (4865, 5, 5), (9729, 3, 5)])             # by the rows: 4, 2, 1
@pytest.mark.parametrize("interp", [0, 1])
def test_adjoint_pass_widths(sep, oracle, rows, npairs, natom, interp):
    print("case adjoint passes", rows, npairs, natom, interp, flush=True)
    grid, d = (16, 24, 16), np.array([0.7, 0.6, 0.8])
    half = 0.5 * d * grid
    rng = np.random.default_rng(rows + npairs)
    dr = np.array([4.0, 3.0, 5.0]) / (rows - 1)
    vr = np.arange(rows)[None, :] * dr[:, None]
    pot = -np.exp(-vr ** 2 / np.array([[2.0], [1.0], [4.0]]))
    npot = np.array([rows, rows - 1, rows])
    xyz = rng.uniform(-0.9, 0.9, (natom, 3)) * half
    types = rng.integers(0, 2, natom).astype(np.int32) * 2  # type 1 has no atoms
    scale = rng.uniform(0.9, 1.1, natom)
    psi = rng.standard_normal((4, int(np.prod(grid))))
    pairs = rng.integers(0, 4, (npairs, 2))
    with sep.Context(*grid, *d, *-half) as ctx:
        ctx.set_interp(interp)
        ctx.states_upload(psi)
        dR, ds, dtab = ctx.hf_adjoint(pairs, xyz, types, npot, vr, pot, dr, scale=scale)
    oracle.set_interp(interp)
    try:
        for p, (i, j) in enumerate(pairs):
            oR, os_, otab = oracle.hf_adjoint(grid, tuple(-half), tuple(d), xyz, types, scale,
                                              npot, vr, pot, dr, psi[i] * psi[j], np.prod(d))
            assert np.abs(dR[p] - oR).max() <= 1e-11 * np.abs(oR).max()
            assert np.abs(ds[p] - os_).max() <= 1e-11 * np.abs(os_).max()
            assert np.abs(dtab[p] - otab).max() <= 1e-11 * np.abs(otab).max()
    finally:
        oracle.set_interp(0)


@pytest.mark.parametrize("rows", [255, 256, 257, 511, 512, 513, 801])
def test_download_pieces(sep, rows):
    """Device to host copies around the 8 MB pieces of the staged path."""
    print("case download", rows, flush=True)
    x = np.random.default_rng(rows).standard_normal((rows, 16 ** 3))  # 32 KB a row
    with sep.Context(16, 16, 16, 0.7, 0.7, 0.7) as ctx:
        ctx.states_upload(x)
        assert np.array_equal(ctx.states_download(rows), x)
        assert np.array_equal(ctx.states_download(rows - 1), x[:-1])  # the halves again
        ctx.trim()
        assert np.array_equal(ctx.states_download(rows), x)
