"""Spinor filters of growing sizes on one context, whose scratch buffer grows
with them: the states of a context that has run smaller filters before are those
of a fresh one, bit for bit, and normalized."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_growing_filters(sep):
    import torch
    n, d = 24, 0.6
    N = n ** 3
    rng = np.random.default_rng(9)
    V = rng.uniform(-1, 1, N)
    xyz, vso = rng.uniform(-5.7, 5.7, (30, 3)), rng.uniform(0.5, 2.0, 30)
    psi = torch.from_numpy(rng.standard_normal((9, 4 * N))).to("cuda:0")
    zn, _ = sep.leja_points(24)

    def context():
        ctx = sep.Context(n, n, n, d, d, d, *((-n * d / 2,) * 3))
        ctx.set_potential(V)
        ctx.so_setup(xyz, vso)
        return ctx

    def run(ctx, ns, ms):
        an = sep.newton_coeffs(zn, np.linspace(-0.5, 0.5, ms), 14.0, -2.0, 4.0)
        ctx.filter_spinor_dev(psi.data_ptr(), ns, an, zn, -2.0, 14.0)
        return ctx.states_download(4 * ns * ms)

    with context() as grown:
        for ns, ms in ((1, 1), (1, 2), (2, 1), (3, 1), (2, 2), (1, 5), (3, 3), (9, 2)):
            print("case spinor scratch", ns, ms, flush=True)
            got = run(grown, ns, ms)
            with context() as fresh:
                ref = run(fresh, ns, ms)
            assert np.array_equal(got, ref)
            norm = (got.reshape(ns * ms, 4 * N) ** 2).sum(1) * d ** 3
            assert np.abs(norm - 1.0).max() < 1e-12
