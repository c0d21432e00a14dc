"""Tiles of the spin-orbit product with stored pair matrices: every
combination of points a lane and spinors a workgroup, with remainders of
both, against the kernel that evaluates the pair expression inline.  Each
point's sums run over q in one order in both, so they agree bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# few atoms / enough atoms for the wider tiles; spinors: one, a full half
# workgroup, one past it, a full workgroup and two uneven groups
@pytest.mark.parametrize("natom,spinors", [(3, (1, 4, 5, 8, 9)), (301, (1, 3, 4, 7)),
                                           (601, (6, 9))])
def test_stored_pairs_match_inline(sep, natom, spinors, monkeypatch):
    import torch
    n, d = 24, 0.55
    rng = np.random.default_rng(natom)
    xyz = rng.uniform(-4.5, 4.5, (natom, 3))
    vso = rng.uniform(0.5, 3.0, natom)
    psi = rng.standard_normal((max(spinors), 4 * n ** 3))
    x = torch.from_numpy(psi).to("cuda:0")
    got = {}
    for knob in ("1", "0"):
        monkeypatch.setenv("SEP_SO_KMAT", knob)
        with sep.Context(n, n, n, d, d, d, *((-n * d / 2,) * 3), ekinmax=20.0) as ctx:
            ctx.set_potential(np.zeros(n ** 3))
            nent = ctx.so_setup(xyz, vso)
            for ns in spinors:
                print(f"case {natom} atoms, {nent / natom:.0f} points, {ns} spinors", flush=True)
                y = torch.empty_like(x[:ns])
                ctx.apply_h_spinor_dev(x.data_ptr(), y.data_ptr(), ns)
                torch.cuda.synchronize()
                got[knob, ns] = y.cpu().numpy()
    for ns in spinors:
        assert np.array_equal(got["1", ns], got["0", ns]), ns
