"""A filter whose ring takes the depth of the 32 GB rule (8 states of 128^3 in
FP64: 256 of 300 Newton vectors, two blocks) against the same filter with blocks
of 96 (hook SEP_RING_DEPTH): the accumulation's sums are blocked differently and
agree to the rounding that 300 steps carry, the bound that FP64 filtered states
are held to against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_blocks_of_the_rule(sep, monkeypatch):
    n, ns, ms, nc = 128, 8, 1, 300
    rng = np.random.default_rng(7)
    print("case ring depth rule", n, ns, ms, nc, flush=True)
    with sep.Context(n, n, n, 0.7, 0.8, 0.9) as ctx:
        ctx.set_potential(rng.uniform(-1.5, 1.0, n ** 3))
        dE, _, _ = ctx.energy_range()
        zn, _ = sep.leja_points(nc)
        an = sep.newton_coeffs(zn, np.linspace(-0.5, 0.5, ms), dE, ctx.vmin,
                               (nc / (2.5 * dE)) ** 2)
        psi0 = rng.standard_normal((ns, n ** 3))
        psi0 /= np.linalg.norm(psi0, axis=1, keepdims=True)
        got, _ = ctx.filter(psi0, an, zn, ctx.vmin, dE, sep.SEP_PREC_FP64)
        monkeypatch.setenv("SEP_RING_DEPTH", "96")
        ref, _ = ctx.filter(psi0, an, zn, ctx.vmin, dE, sep.SEP_PREC_FP64)
    assert np.abs(got - ref).max() <= 1e-9 * np.abs(ref).max()
