"""Orthogonalisation of few states on many points: the double-double Gram
splits the points into as many chunks as fill the GPU (1024 to 65536 points
each), with a ragged last chunk and ragged 16-state tiles.  The singular
values are those of the oracle's SVD to its own rounding (a few eps times the
largest, sqrt(m) more for the reductions), and the kept states orthonormal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 5, 16, 17, 65])
def test_ortho_of_few_states(sep, oracle, m):
    grid, d = (36, 48, 36), 0.7
    print("case ortho chunks", grid, m, flush=True)
    N, dv = int(np.prod(grid)), d ** 3
    rng = np.random.default_rng(m)
    A = rng.standard_normal((m, N))
    if m > 2:  # one direction almost, one exactly contained in the others
        A[1] = A[0] + 1e-6 * A[1]
        A[m - 1] = A[0] - 2.0 * A[1]
    A = oracle.normalize_all(A, dv)
    _, S_o, cut_o = oracle.ortho(A)
    with sep.Context(*grid, d, d, d) as ctx:
        ctx.states_upload(A)
        kept, S = ctx.ortho(m)
        Q = ctx.states_download(kept)
    assert kept == cut_o
    assert np.abs(S - S_o).max() < 1e-13 * S_o[0]
    assert np.abs(Q @ Q.T * dv - np.eye(kept)).max() < 1e-12
