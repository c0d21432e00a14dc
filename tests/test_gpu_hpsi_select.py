"""What sep_set_hpsi_family selects runs, on every grid: the row + strided-line
kernels give the bits of a context opened under the hook that forces them (other
bits than the two-kernel form's, the same H.psi to rounding), the getter names
the family that runs and its answer is accepted, and the autotuner times both.
The chunked and swizzled plane kernels of complex64 128^2 run fused steps and
separate passes alike."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
D = (0.7, 0.8, 0.9)
# grids with and without the plane names; every length, each axis's line kernel
# at the two that no square plane has
GRIDS = [(24, 24, 16), (24, 16, 32), (36, 48, 16), (80, 16, 24), (16, 80, 16), (16, 16, 80),
         (160, 16, 16), (16, 160, 16), (16, 16, 160), (128, 64, 16), (16, 128, 96)]


def _vectors(grid, batch, seed):
    rng = np.random.default_rng(seed)
    N = int(np.prod(grid))
    return (rng.uniform(-1.5, 1.0, N),
            rng.standard_normal((batch, N)) + 1j * rng.standard_normal((batch, N)))


def _apply(sep, ctx, psi, prec):
    if prec == sep.SEP_PREC_FP64:
        return ctx.apply_h(psi)
    import torch
    x = torch.from_numpy(psi.astype(np.complex64)).to("cuda:0")
    y = torch.empty_like(x)
    ctx.apply_h_dev(x.data_ptr(), y.data_ptr(), x.shape[0], prec)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("grid", GRIDS)
def test_lines_run_where_asked_for(sep, oracle, grid, prec, monkeypatch):
    print("case lines", grid, prec, flush=True)
    P = sep.SEP_PREC_FP32 if prec == "fp32" else sep.SEP_PREC_FP64
    V, psi = _vectors(grid, 3, 21)
    named = grid[0] == grid[1]  # PLANE names the two-kernel form
    split = sep.SEP_HPSI_PLANE if named else sep.SEP_HPSI_SPLIT
    with sep.Context(*grid, *D) as ctx:
        ctx.set_potential(V)
        assert ctx.hpsi_family(P) == split
        first = _apply(sep, ctx, psi, P)
        ctx.set_hpsi_family(P, sep.SEP_HPSI_LINES)
        assert ctx.hpsi_family(P) == sep.SEP_HPSI_LINES
        lines = _apply(sep, ctx, psi, P)
        for back in (split, sep.SEP_HPSI_SPLIT):
            ctx.set_hpsi_family(P, sep.SEP_HPSI_LINES)
            ctx.set_hpsi_family(P, back)
            assert ctx.hpsi_family(P) == split
            assert np.array_equal(_apply(sep, ctx, psi, P), first)
        if not named:
            with pytest.raises(RuntimeError):
                ctx.set_hpsi_family(P, sep.SEP_HPSI_PLANE)
            assert ctx.hpsi_family(P) == split
    monkeypatch.setenv("SEP_FORCE_LINE_KERNELS", "1")
    with sep.Context(*grid, *D) as ctx:
        ctx.set_potential(V)
        assert ctx.hpsi_family(P) == sep.SEP_HPSI_LINES
        assert np.array_equal(_apply(sep, ctx, psi, P), lines)
        ctx.set_hpsi_family(P, sep.SEP_HPSI_SPLIT)  # the hook speaks at the opening only
        assert np.array_equal(_apply(sep, ctx, psi, P), first)
    assert not np.array_equal(lines, first)
    ref = oracle.hamiltonian(grid, oracle.ksqr(*grid, *D), V, psi)
    tol = 1e-12 if prec == "fp64" else 2e-6
    for got in (first, lines):
        assert np.abs(got - ref).max() < tol * np.abs(ref).max()


def _filter(sep, ctx, psi0, prec, nc=40, ms=2):
    dE, _, _ = ctx.energy_range()
    zn, _ = sep.leja_points(nc)
    an = sep.newton_coeffs(zn, np.linspace(-0.5, 0.5, ms), dE, ctx.vmin, (nc / (2.5 * dE)) ** 2)
    out, _ = ctx.filter(psi0, an, zn, ctx.vmin, dE, prec)
    return out


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("grid", [(80, 16, 24), (24, 24, 16)])
def test_autotuner_times_both(sep, grid, prec):
    print("case autotune", grid, prec, flush=True)
    P = sep.SEP_PREC_FP32 if prec == "fp32" else sep.SEP_PREC_FP64
    V, psi = _vectors(grid, 4, 22)
    split = sep.SEP_HPSI_PLANE if grid[0] == grid[1] else sep.SEP_HPSI_SPLIT
    with sep.Context(*grid, *D) as ctx:
        ctx.set_potential(V)
        ref = _filter(sep, ctx, psi.real.copy(), P)
        tp, tl = ctx.autotune(P, 2)
        assert tp > 0 and tl > 0
        assert ctx.hpsi_family(P) == (sep.SEP_HPSI_LINES if tl < tp else split)
        ms, fam, lanes = ctx.autotune_ex(P, nvec=2)
        assert {i for i in range(sep.SEP_HPSI_NFAMILY) if ms[i] > 0} == {split, sep.SEP_HPSI_LINES}
        assert ms[fam] == ms[ms > 0].min() and ctx.hpsi_family(P) == fam and lanes in (1, 2)
        for f in (split, sep.SEP_HPSI_LINES):
            ctx.set_hpsi_family(P, f)
            got = _filter(sep, ctx, psi.real.copy(), P)
            err = np.abs(got - ref).max() / np.abs(ref).max()
            print("family", f, "max rel", err, flush=True)
            # the bounds between families of one grid's 40-step filters
            assert err < (1e-5 if prec == "fp32" else 1e-12)


@pytest.mark.parametrize("ns", [3, 8])
@pytest.mark.parametrize("family", ["PLANE_CHUNKED", "PLANE_SWIZZLED"])
def test_plane_forms_fused_equal_separate(sep, family, ns, monkeypatch):
    """The bounds of the default form's fused and separate passes (complex64)."""
    n, P = 128, sep.SEP_PREC_FP32
    print("case fused", family, ns, flush=True)
    rng = np.random.default_rng(23)
    V = rng.uniform(-1.5, 1.0, n ** 3)
    psi0 = rng.standard_normal((ns, n ** 3))
    psi0 /= np.linalg.norm(psi0, axis=1, keepdims=True)
    got = []
    for hook in (False, True):
        if hook:
            monkeypatch.setenv("SEP_SEPARATE_PASSES", "1")
        with sep.Context(n, n, n, *D) as ctx:
            ctx.set_potential(V)
            ctx.set_hpsi_family(P, getattr(sep, "SEP_HPSI_" + family))
            got.append(_filter(sep, ctx, psi0, P))
            if hook:
                ref = _filter(sep, ctx, psi0, sep.SEP_PREC_FP64)
    fused, sepr = got
    scale = np.abs(sepr).max()
    assert np.abs(fused - sepr).max() < 2e-5 * scale
    e_f, e_s = np.abs(fused - ref).max() / scale, np.abs(sepr - ref).max() / scale
    print("vs fp64: fused", e_f, "separate", e_s, flush=True)
    assert e_f <= 1.5 * e_s + 1e-7
