"""The spin-orbit product's tiles for one and two spinors (with three for the
border), few atoms and enough for 64 points a workgroup, list lengths around
whole tiles, against the kernel that evaluates the pair expression inline: bit
for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natom", [1, 9, 145, 147, 300])
@pytest.mark.parametrize("d", [0.55, 0.9])
def test_few_spinors_match_inline(sep, natom, d, monkeypatch):
    import torch
    n = 24
    rng = np.random.default_rng(natom)
    xyz = rng.uniform(-0.4 * n * d, 0.4 * n * d, (natom, 3))
    vso = rng.uniform(0.5, 3.0, natom)
    x = torch.from_numpy(rng.standard_normal((3, 4 * n ** 3))).to("cuda:0")
    got = {}
    for knob in ("1", "0"):
        monkeypatch.setenv("SEP_SO_KMAT", knob)
        with sep.Context(n, n, n, d, d, d, *((-n * d / 2,) * 3), ekinmax=20.0) as ctx:
            ctx.set_potential(np.zeros(n ** 3))
            nent = ctx.so_setup(xyz, vso)
            for ns in (1, 2, 3):
                print(f"case {natom} atoms, {nent / natom:.0f} points, {ns} spinors", flush=True)
                y = torch.empty_like(x[:ns])
                ctx.apply_h_spinor_dev(x.data_ptr(), y.data_ptr(), ns)
                torch.cuda.synchronize()
                got[knob, ns] = y.cpu().numpy()
    for ns in (1, 2, 3):
        assert np.array_equal(got["1", ns], got["0", ns]), ns
