"""The two-kernel H.psi (csrc/sep_split.h) against the CPU oracle where it can
go wrong: every y plan (4, 6, 8 and 16 rows a group) with x lengths shorter and
longer than a group's rows, workgroups that hold several pairs of groups with
a ragged last one ((16, 80, 36): 90 pairs, 4 a workgroup), tiles whose z lines
do not fill the threads' last round, and the three forms of a vector
(interleaved, two real planes, one real plane).  Rounding of a three-pass FFT
of 10^6 points stays below 1e-14 (FP64) and 2e-6 (complex64) of the largest
value; the filter's 16 Newton steps amplify it by at most 2e2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRIDS = [(16, 16, 16), (16, 80, 36), (128, 16, 24), (24, 128, 16), (36, 36, 36), (48, 64, 80),
         (80, 24, 160), (160, 36, 32), (64, 160, 16), (32, 96, 48), (96, 48, 128),
         (16, 96, 96), (24, 160, 80), (16, 160, 160)]


@pytest.mark.parametrize("grid", GRIDS)
def test_split_forms_vs_oracle(sep, oracle, grid):
    import torch
    nx, ny, nz = grid
    print("case split", grid, flush=True)
    rng = np.random.default_rng(nx * 7 + ny * 3 + nz)
    d = (0.7, 0.8, 0.9)
    N = nx * ny * nz
    ksq = oracle.ksqr(nx, ny, nz, *d)
    pot = rng.uniform(-1.5, 1.0, N)
    x = rng.standard_normal((3, N))
    with sep.Context(nx, ny, nz, *d) as ctx:
        ctx.set_potential(pot)
        # interleaved, both precisions
        z = x[:2] + 1j * x[1:]
        ref = oracle.hamiltonian(grid, ksq, pot, z)
        scale = np.abs(ref).max()
        assert np.abs(ctx.apply_h(z) - ref).max() < 1e-13 * scale
        c = torch.from_numpy(z.astype(np.complex64)).to("cuda:0")
        o = torch.empty_like(c)
        ctx.apply_h_dev(c.data_ptr(), o.data_ptr(), 2, sep.SEP_PREC_FP32)
        assert np.abs(o.cpu().numpy() - ref).max() < 2e-6 * scale
        # two planes and one plane (odd number of states), with the sums
        ctx.states_upload(x)
        hx = oracle.hamiltonian(grid, ksq, pot, x.astype(np.complex128)).real
        e = (x * hx).sum(axis=1) * ctx.dv
        assert np.abs(ctx.energy_all(3) - e).max() < 1e-12 * np.abs(e).max()
        # the filter's fused steps (odd: the last vector's second plane is zero)
        nc = 17
        an = 1.0 / (1.0 + np.arange(nc))[None, :]
        zn = np.cos(np.pi * np.arange(nc) / nc)
        vmin, dE = -1.5, 24.0
        want, p = np.zeros_like(x), x.copy()
        for j in range(nc):
            if j:
                hp = oracle.hamiltonian(grid, ksq, pot, p.astype(np.complex128)).real
                p = 4.0 / dE * hp - (2.0 + zn[j - 1] + vmin * 4.0 / dE) * p
            want += an[0, j] * p
        want /= np.sqrt((want * want).sum(axis=1, keepdims=True) * ctx.dv)
        for prec, tol in ((sep.SEP_PREC_FP64, 2e-12), (sep.SEP_PREC_FP32, 4e-4)):
            got, _ = ctx.filter(x, an, zn, vmin, dE, prec, want_energies=False)
            assert np.abs(got - want).max() < tol * np.abs(want).max(), prec
