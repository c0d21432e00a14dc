"""Performance cases of the filter-diagonalization library.

Each case is one call (or the short sequence of calls) that a program built on
semi_empirical_pseudopotentials_amd makes: H.psi on device vectors, the
spectral range, V(r), the Newton filter, the subspace stage, the spin-orbit H
and the Hellmann-Feynman adjoint.  Sizes are those of the repository's tests,
decks and benchmark, from the 16^3 grid of the smallest tests to 160^3.

prepare() opens the context (grid, potential, lists) and makes the inputs a
program holds before the call; run() is the call; exact() restates it in
64 bits with torch alone.
"""
import functools
import math

import numpy as np
import torch

import semi_empirical_pseudopotentials_amd as sep
from semi_empirical_pseudopotentials_amd import decks

DEV = "cuda:0"
LENGTHS = (16, 24, 32, 36, 48, 64, 80, 96, 128, 160)
FP64, FP32 = sep.SEP_PREC_FP64, sep.SEP_PREC_FP32
# spin-orbit strengths of In and As in Ha (a = 6.057 A)
VSO = {"In": 0.48 * (6.057 / 0.529177) ** 3 / 8.0 / 27.2114, "As": 3.15164354}


def listed():
    return [
        # one H.psi on the smallest test grid: the latency of a single call,
        # as in an outer eigensolver's inner loop
        {"name": "apply_16_c128", "kind": "apply", "nx": 16, "ny": 16, "nz": 16, "bits": 64,
         "batch": 1, "dot": 1.2},
        # the non-cubic box of the 2.2 nm CdSe deck, an odd number of vectors
        {"name": "apply_80x64x64_c128", "kind": "apply", "nx": 80, "ny": 64, "nz": 64, "bits": 64,
         "batch": 5, "dot": 2.2},
        # the largest grid, a block of vectors in single precision
        {"name": "apply_160_c64", "kind": "apply", "nx": 160, "ny": 160, "nz": 160, "bits": 32,
         "batch": 8, "dot": 5.0},
        # the spectral bound every run starts with: H.psi on one vector, in turn
        {"name": "range_64", "kind": "range", "nx": 64, "ny": 64, "nz": 64, "dot": 2.0},
        # V(r) of the 4 nm dot: once per geometry in a relaxation or a fit
        {"name": "potential_128", "kind": "potential", "nx": 128, "ny": 128, "nz": 128, "dot": 4.0,
         "cubic": False},
        # the In13_P16 deck's filter: 10 targets x 16 states, Newton length 1024
        {"name": "filter_36_c128", "kind": "filter", "nx": 36, "ny": 36, "nz": 36, "bits": 64,
         "ns": 16, "ms": 10, "nc": 1024, "dot": 1.2},
        # 2 nm dot at 64^3, 8 targets x 4 states, single-precision recurrence
        {"name": "filter_64_c64", "kind": "filter", "nx": 64, "ny": 64, "nz": 64, "bits": 32,
         "ns": 4, "ms": 8, "nc": 192, "dot": 2.0},
        # 4 nm dot at 128^3, one target at a time, both precisions
        {"name": "filter_128_c64", "kind": "filter", "nx": 128, "ny": 128, "nz": 128, "bits": 32,
         "ns": 16, "ms": 1, "nc": 192, "dot": 4.0},
        {"name": "filter_128_c128", "kind": "filter", "nx": 128, "ny": 128, "nz": 128, "bits": 64,
         "ns": 8, "ms": 1, "nc": 512, "dot": 4.0},
        # spin-orbit H of the 3 nm InAs dot at 96^3 on a block of spinors
        {"name": "spinor_96", "kind": "spinor", "nx": 96, "ny": 96, "nz": 96, "ns": 8, "dot": 3.0},
        # filter, ortho, Rayleigh-Ritz and sigma of a 1.5 nm dot in one go
        {"name": "levels_48", "kind": "levels", "nx": 48, "ny": 48, "nz": 48, "ns": 16, "ms": 4,
         "nc": 192, "dot": 1.5},
        # backward: forces and table gradients of 8 levels, 3 nm dot at 96^3
        {"name": "adjoint_96", "kind": "adjoint", "nx": 96, "ny": 96, "nz": 96, "pairs": 8,
         "weighted": False, "dot": 3.0, "cubic": False},
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["apply", "apply", "range", "potential", "filter", "filter", "filter",
                       "spinor", "levels", "adjoint"])
    top = {"apply": 160, "range": 96, "potential": 128, "filter": 128, "spinor": 96, "levels": 64,
           "adjoint": 96}[kind]
    low = 16 if kind == "apply" else 24
    sizes = [n for n in LENGTHS if low <= n <= top]
    n = rng.choice(sizes)
    c = {"kind": kind, "nx": n, "ny": n, "nz": n}
    if kind != "spinor" and rng.random() < 0.35:  # a box longer on some axes
        near = [m for m in sizes if n / 2 <= m <= n]
        c["ny"], c["nz"] = rng.choice(near), rng.choice(near)
    N = c["nx"] * c["ny"] * c["nz"]
    c["dot"] = round(min(4.5, max(1.2, n / 32.0) * rng.uniform(0.9, 1.1)), 2)
    if kind == "apply":
        c["bits"] = rng.choice([32, 64])
        c["batch"] = _spread(rng, 1, max(1, min(48, 8 * 160 ** 3 // N)))
    elif kind in ("potential", "adjoint"):
        c["cubic"] = rng.random() < 0.4
        if kind == "adjoint":
            c["weighted"] = rng.random() < 0.5
            c["pairs"] = _spread(rng, 1, 12)
    elif kind == "filter":
        c["bits"] = rng.choice([32, 64])
        c["ns"] = _spread(rng, 1, max(2, min(24, 8 * 128 ** 3 // N)))
        c["ms"] = _spread(rng, 1, max(2, min(12, 12 * 128 ** 3 // (N * c["ns"]))))
        # single precision: short filters, whose states agree to 2e-5 however
        # the recurrence is rounded (a longer one carries more of its noise)
        most = 1024 * 96 ** 3 * 8 // (N * c["ns"])
        c["nc"] = _spread(rng, 48, max(64, min(1024 if c["bits"] == 64 else 192, most)))
    elif kind == "spinor":
        c["ns"] = _spread(rng, 1, 8)
    elif kind == "levels":
        c["ns"] = rng.randint(6, 20)
        c["ms"] = rng.randint(1, 4)
        c["nc"] = _spread(rng, 64, 256)
    return c


# ------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def _sites(dot):
    syms, xyz = decks.cdse_dot(dot)
    return syms, xyz - xyz.mean(axis=0)


def _atoms(case, seed):
    """Symbols and positions of the dot, each atom displaced as by a relaxation."""
    syms, xyz = _sites(case["dot"])
    xyz = xyz + np.random.default_rng(seed).uniform(-0.05, 0.05, xyz.shape)
    return syms, xyz - xyz.mean(axis=0)


def _box(case, seed):
    syms, xyz = _atoms(case, seed)
    half, d = decks.box_from_atoms(xyz, case["nx"], case["ny"], case["nz"])
    return syms, xyz, half, d


def _tables(dr=0.01):
    """Radial tables of Cd, Se and the two ligands, shifted to 0 at the last row."""
    names = ("Cd", "Se", "P1", "P2")
    rows = [decks.pot_table(*decks.DEFAULT_POTS[s], dr=dr) for s in names]
    vr = np.array([r for r, _ in rows])
    pot = np.array([v - v[-1] for _, v in rows])
    return (names, vr, pot, np.full(4, vr.shape[1], dtype=np.int64),
            np.array([r[1] - r[0] for r, _ in rows]))


def _axes(case, half, d):
    return [torch.arange(n, dtype=torch.float64, device=DEV) * float(d[a]) - float(half[a])
            for a, n in enumerate((case["nx"], case["ny"], case["nz"]))]


def _wells(case, seed):
    """(V as an N-vector on the device, half box, spacing): the sum of the
    dot's Gaussian wells, as products of its axes."""
    syms, xyz, half, d = _box(case, seed)
    x, y, z = _axes(case, half, d)
    V = torch.zeros((case["nz"], case["ny"] * case["nx"]), dtype=torch.float64, device=DEV)
    for s in sorted(set(syms)):
        R = torch.tensor(xyz[[t == s for t in syms]], dtype=torch.float64, device=DEV)
        A, sg, B, tau = decks.DEFAULT_POTS[s]
        for amp, w in ((A, sg), (B, tau)):
            if amp == 0.0:
                continue
            g = [torch.exp(-((t[None, :] - R[:, a:a + 1]) / w) ** 2)
                 for a, t in enumerate((x, y, z))]
            xy = (g[1][:, :, None] * g[0][:, None, :]).reshape(R.shape[0], -1)
            V += amp * (g[2].t().contiguous() @ xy)
    return V.reshape(-1), half, d


def _open(case, half, d, ekinmax=10.0):
    return sep.Context(case["nx"], case["ny"], case["nz"], float(d[0]), float(d[1]), float(d[2]),
                       -float(half[0]), -float(half[1]), -float(half[2]), ekinmax=ekinmax)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) % (1 << 31))


def _random_states(m, N, dv, seed):
    """Uniform [-1, 1] random states, each normalized."""
    psi = torch.empty((m, N), dtype=torch.float64, device=DEV).uniform_(-1.0, 1.0,
                                                                        generator=_gen(seed))
    return psi / torch.sqrt((psi * psi).sum(dim=1, keepdim=True) * dv)


@functools.lru_cache(maxsize=None)
def _leja(nc):
    return sep.leja_points(nc)[0]


def _newton(case, V):
    """Newton points and coefficients of the case's targets, energies inside
    the spectrum (the dots' levels start a little above 0), on [Vmin, Vmin + dE]."""
    vmin = float(V.min())
    dE = 1.1 * (10.0 + float(V.max()) - vmin)
    el = np.linspace(0.1, 0.5, case["ms"])
    zn = _leja(case["nc"])
    an = sep.newton_coeffs(zn, el, dE, vmin, (case["nc"] / (2.5 * dE)) ** 2)
    return vmin, dE, zn, an


def _potential_args(case, seed):
    syms, xyz, half, d = _box(case, seed)
    names, vr, pot, npot, dr = _tables()
    types = np.array([names.index(s) for s in syms], dtype=np.int32)
    scale = np.random.default_rng(seed + 1).uniform(0.98, 1.02, len(syms))
    return (xyz, types, npot, vr, pot, dr, scale), half, d


def _smooth_states(case, half, d, m, seed):
    """m normalized states that fall off towards the faces of the box."""
    x, y, z = _axes(case, half, d)
    env = (torch.cos(0.5 * math.pi * z / float(half[2]))[:, None, None] *
           torch.cos(0.5 * math.pi * y / float(half[1]))[None, :, None] *
           torch.cos(0.5 * math.pi * x / float(half[0]))[None, None, :]).reshape(-1)
    psi = env * torch.randn((m, env.numel()), dtype=torch.float64, device=DEV, generator=_gen(seed))
    return psi / torch.sqrt((psi * psi).sum(dim=1, keepdim=True) * float(np.prod(d)))


def _so_atoms(case, seed):
    syms, xyz, half, d = _box(case, seed)
    vso = np.array([VSO.get({"Cd": "In", "Se": "As"}.get(s, s), 0.0) for s in syms])
    return xyz, vso, half, d


def prepare(case, seed):
    k = case["kind"]
    N = case["nx"] * case["ny"] * case["nz"]
    if k in ("potential", "adjoint"):
        args, half, d = _potential_args(case, seed)
        ctx = _open(case, half, d)
        ctx.set_interp(sep.SEP_INTERP_CUBIC if case["cubic"] else sep.SEP_INTERP_LINEAR)
        st = {"kind": k, "ctx": ctx, "args": args}
        if k == "adjoint":
            m = max(2, case["pairs"])
            ctx.states_upload(_smooth_states(case, half, d, m, seed).cpu().numpy())
            i = np.arange(case["pairs"])
            # levels' own densities, then couplings of neighbours
            st["pairs"] = np.stack([i % m, np.where(i % 3 == 2, (i + 1) % m, i % m)], axis=1)
            st["w"] = (np.random.default_rng(seed).uniform(-1.0, 1.0, case["pairs"])
                       if case["weighted"] else None)
        return st
    if k == "spinor":
        xyz, vso, half, d = _so_atoms(case, seed)
        V = _wells(case, seed)[0]
        ctx = _open(case, half, d, ekinmax=20.0)
        ctx.set_potential(V.cpu().numpy())
        ctx.so_setup(xyz, vso)
        x = torch.randn((case["ns"], 4, N), dtype=torch.float64, device=DEV, generator=_gen(seed))
        return {"kind": k, "ctx": ctx, "in": x, "out": torch.empty_like(x), "ns": case["ns"]}
    V, half, d = _wells(case, seed)
    ctx = _open(case, half, d)
    ctx.set_potential(V.cpu().numpy())
    st = {"kind": k, "ctx": ctx}
    if k == "apply":
        dt = torch.complex128 if case["bits"] == 64 else torch.complex64
        x = torch.randn((case["batch"], N), dtype=dt, device=DEV, generator=_gen(seed))
        st.update({"in": x, "out": torch.empty_like(x), "batch": case["batch"],
                   "prec": FP64 if case["bits"] == 64 else FP32})
    elif k in ("filter", "levels"):
        st["newton"] = _newton(case, V)
        st["psi0"] = _random_states(case["ns"], N, float(np.prod(d)), seed)
        st["ns"], st["m"] = case["ns"], case["ns"] * case["ms"]
        st["single"] = case.get("bits", 64) == 32
    return st


# ------------------------------------------------------------------ the calls
def run(st):
    ctx, k = st["ctx"], st["kind"]
    if k == "apply":
        ctx.apply_h_dev(st["in"].data_ptr(), st["out"].data_ptr(), st["batch"], st["prec"])
        return st["out"]
    if k == "spinor":
        ctx.apply_h_spinor_dev(st["in"].data_ptr(), st["out"].data_ptr(), st["ns"])
        return st["out"]
    if k == "range":
        dE, emax, iters = ctx.energy_range()
        return {"dE": dE, "emax": emax, "iters": iters}
    if k == "potential":
        xyz, types, npot, vr, pot, dr, scale = st["args"]
        V = ctx.build_potential(xyz, types, npot, vr, pot, dr, scale=scale)
        return {"V": V, "vmin": ctx.vmin, "vmax": ctx.vmax}
    if k == "adjoint":
        xyz, types, npot, vr, pot, dr, scale = st["args"]
        dR, ds, dtab = ctx.hf_adjoint(st["pairs"], xyz, types, npot, vr, pot, dr, scale=scale,
                                      weights=st["w"])
        return {"dR": dR, "dscale": ds, "dtab": dtab}
    vmin, dE, zn, an = st["newton"]
    ctx.filter_dev(st["psi0"].data_ptr(), st["ns"], an, zn, vmin, dE,
                   FP32 if st["single"] else FP64)
    if k == "filter":
        psi = ctx.states_download(st["m"])
        # states of the single-precision recurrence are kept in its precision
        return torch.from_numpy(psi).float() if st["single"] else psi
    kept, S = ctx.ortho(st["m"])
    ev = ctx.rayleigh_ritz(kept)
    sg = ctx.sigma(kept)
    return {"kept": kept, "S": S, "ev": ev, "sigma": sg, "psi": ctx.states_download(kept)}


def work(case):
    k = case["kind"]
    N = case["nx"] * case["ny"] * case["nz"]
    fft = 2 * 5 * N * math.log2(N)  # forward and inverse, per complex vector
    if k == "apply":
        b = case["bits"] // 8
        return {"bytes": N * (case["batch"] * 4 * b + b), "flops": case["batch"] * (fft + 8 * N)}
    if k == "spinor":
        return {"bytes": N * (case["ns"] * 64 + 8), "flops": 2 * case["ns"] * (fft + 8 * N)}
    if k == "range":
        return {"bytes": 24 * N, "flops": 20 * (fft + 12 * N)}
    atoms = len(_sites(case["dot"])[0])
    if k == "potential":
        return {"bytes": 8 * N, "flops": 60 * N}
    if k == "adjoint":
        out = 1 if case["weighted"] else case["pairs"]
        return {"bytes": 8 * N * max(2, case["pairs"]) + 8 * out * (4 * atoms + 4 * 1201),
                "flops": 100 * N * out}
    nvec = (case["ns"] + 1) // 2
    m = case["ns"] * case["ms"]
    steps = case["nc"] - 1
    f = {"bytes": 8 * N * (case["ns"] + m), "flops": steps * (nvec * (fft + 12 * N) + 2 * m * N)}
    if k == "levels":
        f["flops"] += 10 * m * m * N + m * fft
    return f


# ------------------------------------------------------------------ 64-bit values
def _ksq(case, d, ekinmax):
    n3 = (case["nx"], case["ny"], case["nz"])
    k2 = []
    for n, h in zip(n3, d):
        j = torch.arange(n, dtype=torch.float64, device=DEV)
        j = torch.minimum(j, n - j)
        k2.append(0.5 * (j * (2.0 * math.pi / (n * float(h)))) ** 2)
    t = k2[2][:, None, None] + k2[1][None, :, None] + k2[0][None, None, :]
    return torch.clamp(t, max=ekinmax)


def _h(case, kin, V, z):
    """H on complex128 vectors (rows of z)."""
    g = z.reshape(-1, case["nz"], case["ny"], case["nx"])
    t = torch.fft.ifftn(torch.fft.fftn(g, dim=(1, 2, 3)) * kin, dim=(1, 2, 3))
    return t.reshape(z.shape) + V * z


def _filtered(case, seed):
    """The filter's normalized states, and what they were made with."""
    V, half, d = _wells(case, seed)
    N, dv = V.numel(), float(np.prod(d))
    vmin, dE, zn, an = _newton(case, V)
    psi0 = _random_states(case["ns"], N, dv, seed)
    nv = (case["ns"] + 1) // 2
    z = torch.zeros((nv, N), dtype=torch.complex128, device=DEV)
    z.real.copy_(psi0[0::2])
    z.imag[:case["ns"] // 2].copy_(psi0[1::2])
    kin = _ksq(case, d, 10.0)
    acc = torch.zeros((case["ns"], case["ms"], N), dtype=torch.float64, device=DEV)
    coef = torch.tensor(an, dtype=torch.float64, device=DEV)
    for j in range(case["nc"]):
        if j > 0:
            z = (4.0 / dE) * _h(case, kin, V, z) - (2.0 + zn[j - 1] + vmin * 4.0 / dE) * z
        for s in range(case["ns"]):
            row = z[s // 2].real if s % 2 == 0 else z[s // 2].imag
            if case["ms"] == 1:
                acc[s, 0] += an[0, j] * row
            else:
                acc[s].addcmul_(coef[:, j:j + 1], row[None, :])
    acc = acc.reshape(-1, N)
    acc /= torch.sqrt((acc * acc).sum(dim=1, keepdim=True) * dv)
    return acc, V, kin, dv


def _segments(case, args, half, d):
    """Per atom: grid indices of its box, distances, offsets and table segment."""
    xyz, types, npot, vr, pot, dr, scale = args
    ax = _axes(case, half, d)
    for a in range(len(types)):
        t = int(types[a])
        rmax = (int(npot[t]) - 1) * float(dr[t])
        sub = [torch.nonzero((q - float(xyz[a, i])).abs() <= rmax).reshape(-1)
               for i, q in enumerate(ax)]
        dx, dy, dz = (ax[i][sub[i]] - float(xyz[a, i]) for i in range(3))
        r = torch.sqrt(dz[:, None, None] ** 2 + dy[None, :, None] ** 2 + dx[None, None, :] ** 2)
        g = ((sub[2][:, None, None] * case["ny"] + sub[1][None, :, None]) * case["nx"] +
             sub[0][None, None, :]).expand(r.shape)
        off = [q.expand(r.shape) for q in (dx[None, None, :], dy[None, :, None], dz[:, None, None])]
        i = (r / float(dr[t])).long()
        ok = i <= int(npot[t]) - 2
        yield a, t, g[ok], r[ok], [o[ok] for o in off], i[ok]


def _row_weights(cubic, n, i, w):
    """Table rows and their weights (and derivatives in w) of the interpolant."""
    if not cubic:
        one = torch.ones_like(w)
        return [i, i + 1], [1.0 - w, w], [-one, one]
    h = [2 * w ** 3 - 3 * w ** 2 + 1, w ** 3 - 2 * w ** 2 + w, -2 * w ** 3 + 3 * w ** 2,
         w ** 3 - w ** 2]
    g = [6 * w ** 2 - 6 * w, 3 * w ** 2 - 4 * w + 1, -6 * w ** 2 + 6 * w, 3 * w ** 2 - 2 * w]
    # tangents: half the difference of the neighbours, one-sided at the ends
    first, last = (i == 0), (i == n - 2)
    rows = [torch.clamp(i - 1, min=0), i, i + 1, torch.clamp(i + 2, max=n - 1)]
    ws = []
    for p0, m0, p1, m1 in (h, g):
        a0 = torch.where(first, torch.zeros_like(w), -0.5 * m0)
        a1 = p0 + torch.where(first, -m0, torch.zeros_like(w)) - \
            torch.where(last, m1, 0.5 * m1)
        a2 = p1 + torch.where(first, m0, 0.5 * m0) + torch.where(last, m1, torch.zeros_like(w))
        a3 = torch.where(last, torch.zeros_like(w), 0.5 * m1)
        ws.append([a0, a1, a2, a3])
    return rows, ws[0], ws[1]


def _exact_potential(case, seed):
    args, half, d = _potential_args(case, seed)
    xyz, types, npot, vr, pot, dr, scale = args
    V = torch.zeros(case["nx"] * case["ny"] * case["nz"], dtype=torch.float64, device=DEV)
    vr_t, pot_t = (torch.tensor(q, device=DEV) for q in (vr, pot))
    for a, t, g, r, off, i in _segments(case, args, half, d):
        w = (r - vr_t[t][i]) / (vr_t[t][i + 1] - vr_t[t][i])
        rows, ws, _ = _row_weights(case["cubic"], int(npot[t]), i, w)
        V[g] += float(scale[a]) * sum(q * pot_t[t][k] for k, q in zip(rows, ws))
    return {"V": V.cpu().numpy(), "vmin": float(V.min()), "vmax": float(V.max())}


def _exact_adjoint(case, seed):
    st_args, half, d = _potential_args(case, seed)
    xyz, types, npot, vr, pot, dr, scale = st_args
    m, dv = max(2, case["pairs"]), float(np.prod(d))
    psi = _smooth_states(case, half, d, m, seed)
    i = np.arange(case["pairs"])
    j = np.where(i % 3 == 2, (i + 1) % m, i % m)
    rho = psi[torch.tensor(i % m, device=DEV)] * psi[torch.tensor(j, device=DEV)]
    if case["weighted"]:
        w = np.random.default_rng(seed).uniform(-1.0, 1.0, case["pairs"])
        rho = (torch.tensor(w, device=DEV)[:, None] * rho).sum(dim=0, keepdim=True)
    P, na = rho.shape[0], len(types)
    dR = torch.zeros((P, na, 3), dtype=torch.float64, device=DEV)
    ds = torch.zeros((P, na), dtype=torch.float64, device=DEV)
    dt = torch.zeros((P,) + vr.shape, dtype=torch.float64, device=DEV)
    vr_t, pot_t = (torch.tensor(q, device=DEV) for q in (vr, pot))
    for a, t, g, r, off, k in _segments(case, st_args, half, d):
        span = vr_t[t][k + 1] - vr_t[t][k]
        rows, ws, dw = _row_weights(case["cubic"], int(npot[t]), k, (r - vr_t[t][k]) / span)
        val = sum(q * pot_t[t][n] for n, q in zip(rows, ws))
        slope = sum(q * pot_t[t][n] for n, q in zip(rows, dw)) / span
        f = torch.where(r > 0, -float(scale[a]) * slope / torch.clamp(r, min=1e-300),
                        torch.zeros_like(r))
        rg = rho[:, g]
        for c in range(3):
            dR[:, a, c] = (rg * (f * off[c])).sum(dim=1) * dv
        ds[:, a] = (rg * val).sum(dim=1) * dv
        for n, q in zip(rows, ws):
            dt[:, t].index_add_(1, n, rg * (q * (float(scale[a]) * dv)))
    return {"dR": dR.cpu().numpy(), "dscale": ds.cpu().numpy(), "dtab": dt.cpu().numpy()}


def _exact_spinor(case, seed):
    """(T + V + V_so) psi, the nonlocal term atom by atom as dense pair kernels."""
    xyz, vso, half, d = _so_atoms(case, seed)
    V = _wells(case, seed)[0]
    N, dv, sigma = V.numel(), float(np.prod(d)), float(d[0])
    x = torch.randn((case["ns"], 4, N), dtype=torch.float64, device=DEV, generator=_gen(seed))
    psi = torch.complex(x[:, 0::2].contiguous(), x[:, 1::2].contiguous())  # (ns, 2, N)
    out = _h(case, _ksq(case, d, 20.0), V, psi)
    ax = _axes(case, half, d)
    cut = 0.49 * 6.0 * math.log(10.0)
    c = 0.5 / math.sqrt(2.0 * math.pi * sigma * sigma) * dv
    r2 = math.sqrt(2.0)
    for a in np.nonzero(vso)[0]:
        sub = [torch.nonzero((q - float(xyz[a, i])) ** 2 < cut).reshape(-1)
               for i, q in enumerate(ax)]
        dx, dy, dz = (ax[i][sub[i]] - float(xyz[a, i]) for i in range(3))
        shape = (dz.numel(), dy.numel(), dx.numel())
        dx, dy, dz = (q.expand(shape) for q in (dx[None, None, :], dy[None, :, None],
                                                dz[:, None, None]))
        q2 = dx * dx + dy * dy + dz * dz
        ok = q2 < cut
        g = ((sub[2][:, None, None] * case["ny"] + sub[1][None, :, None]) * case["nx"] +
             sub[0][None, None, :])[ok]
        dx, dy, dz, q2 = dx[ok], dy[ok], dz[ok], q2[ok]
        r = torch.sqrt(q2)
        v = float(vso[a]) * torch.exp(-q2 / 0.49)
        K = (v[:, None] + v[None, :]) * torch.exp(-0.5 * ((r[:, None] - r[None, :]) / sigma) ** 2)
        K = (K / (q2[:, None] + q2[None, :])).to(torch.complex128)
        n1, n0 = math.sqrt(3.0 / (8.0 * math.pi)), math.sqrt(3.0 / (4.0 * math.pi))
        y = {1: torch.complex(-n1 * dx / r, -n1 * dy / r), 0: torch.complex(n0 * dz / r, 0 * r),
             -1: torch.complex(n1 * dx / r, -n1 * dy / r)}
        S = {m: [(q.conj() * psi[:, s, g]) @ K for s in (0, 1)] for m, q in y.items()}
        out[:, 0, g] += c * (y[1] * S[1][0] - y[-1] * S[-1][0] +
                             r2 * (y[0] * S[1][1] + y[-1] * S[0][1]))
        out[:, 1, g] += c * (-y[1] * S[1][1] - y[-1] * S[-1][1] +
                             r2 * (y[0] * S[-1][0] + y[1] * S[0][0]))
    res = torch.empty_like(x)
    res[:, 0::2], res[:, 1::2] = out.real, out.imag
    return res


def exact(case, seed):
    k = case["kind"]
    if k == "range":
        return None  # its start vector is the library's own random stream
    if k == "potential":
        return _exact_potential(case, seed)
    if k == "adjoint":
        return _exact_adjoint(case, seed)
    if k == "spinor":
        return _exact_spinor(case, seed)
    if k == "apply":
        V, half, d = _wells(case, seed)
        dt = torch.complex128 if case["bits"] == 64 else torch.complex64
        x = torch.randn((case["batch"], V.numel()), dtype=dt, device=DEV, generator=_gen(seed))
        kin = _ksq(case, d, 10.0)
        return torch.cat([_h(case, kin, V, v[None].to(torch.complex128)) for v in x])
    A, V, kin, dv = _filtered(case, seed)
    if k == "filter":
        return A.cpu()
    S = torch.linalg.svdvals(A.t().contiguous().cpu()).numpy()
    Q = torch.linalg.qr(A.t().contiguous().cpu())[0].t().contiguous().to(DEV)  # rows orthonormal
    HQ = torch.cat([_h(case, kin, V, q[None].to(torch.complex128)).real for q in Q])
    P = (Q @ HQ.t().contiguous()).cpu()
    ev, W = torch.linalg.eigh(0.5 * (P + P.t()))
    HR = W.t().contiguous().to(DEV) @ HQ
    sg = torch.sqrt(torch.abs((HR * HR).sum(dim=1).cpu() - ev * ev))
    # Ritz vectors are fixed up to a sign each: no value for them
    return {"kept": None, "S": S, "ev": ev.numpy(), "sigma": sg.numpy(), "psi": None}
