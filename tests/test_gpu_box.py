"""H.psi of a vector held by one CU (csrc/sep_box.hip) against the CPU oracle:
every grid of the form and its nearest neighbours outside it, the three forms
of a vector (interleaved, two real planes, one real plane), in place, with the
epilogue's sums, and at 1 and 65 vectors.  A three-axis FFT of 6144 points
rounds below 1e-14 (FP64) and 2e-6 (complex64) of the largest value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(16, 16, 16), (24, 16, 16), (16, 24, 16), (16, 16, 24),
                                  (24, 24, 16), (16, 32, 16)])
def test_one_kernel_apply_vs_oracle(sep, oracle, grid):
    import torch
    nx, ny, nz = grid
    rng = np.random.default_rng(nx + 3 * ny + 7 * nz)
    d = (0.7, 0.8, 0.9)
    N = nx * ny * nz
    ksq = oracle.ksqr(nx, ny, nz, *d)
    pot = rng.uniform(-1.5, 1.0, N)
    z = rng.standard_normal((65, N)) + 1j * rng.standard_normal((65, N))
    x = np.ascontiguousarray(z.real[:5])
    ref = oracle.hamiltonian(grid, ksq, pot, z)
    hx = oracle.hamiltonian(grid, ksq, pot, x.astype(np.complex128)).real
    scale = np.abs(ref).max()
    with sep.Context(nx, ny, nz, *d) as ctx:
        ctx.set_potential(pot)
        for n in (1, 65):
            print("case one kernel", grid, n, flush=True)
            assert np.abs(ctx.apply_h(z[:n]) - ref[:n]).max() < 1e-13 * scale
            c = torch.from_numpy(z[:n].astype(np.complex64)).to("cuda:0")
            ctx.apply_h_dev(c.data_ptr(), c.data_ptr(), n, sep.SEP_PREC_FP32)  # in place
            assert np.abs(c.cpu().numpy() - ref[:n]).max() < 2e-6 * scale
        # planes: pairs of real states, and the odd last one alone, with the sums
        ctx.states_upload(x)
        e = (x * hx).sum(axis=1) * ctx.dv
        assert np.abs(ctx.energy_all(5) - e).max() < 1e-12 * np.abs(e).max()
