"""The work a user of this package has it do, as timed and checked cases.

Three kinds, each through the package's public entry points:

  minimise  one fixed-ion electronic minimisation on a `CPContext`: the
            coefficients go in, some steps run (steepest descent or conjugate
            gradient, V(r) fixed or rebuilt from each step's density, with or
            without the non-local projectors), the energies of the last step
            and the coefficients come back;
  serve     a mix of independent minimisations of different sizes submitted to
            one `serve.Server` and drained;
  ortho     the stateless (S/2)^{-1/2} of a host matrix.

The systems are water boxes at the density of 32 molecules in 9.86 A, four
states per molecule, 30 to 70 Ry, on the smallest grid with compiled transforms
that holds the density sphere.  A real minimisation takes a few hundred steps;
a pass runs 25 to 100 so that it stays short.

Results of mixed precision contexts come out of single precision transforms
and are returned at single precision; all others are double.
"""
import functools
import math

import numpy as np
import torch

from openatom_amd import _lib, serve, system
from openatom_amd.step import CPContext

# time steps (a.u.): steepest descent as in the benchmark, conjugate gradient
# as in the request loop
DT = {"sd": 5.0, "cg": 160.0}
BOHR = system.BOHR_PER_ANG
PAD = 0.02  # density sphere components closer than this to the next integer still fit


def listed():
    m = functools.partial(dict, kind="minimise", shape="cubic", nonlocal_kb=False, resid=False,
                          monitor=False, autotune=False)
    return [
        # the stateless orthonormalisation a host code calls on its own S: the smallest call
        dict(name="ortho-48", kind="ortho", n=48),
        # ... and for as many states as the 64-molecule requests have
        dict(name="ortho-256", kind="ortho", n=256),
        # the smallest requests: a few molecules, every step's |F| read back
        m(name="water4-mixed-cg", nmol=4, ecut=50.0, precision="mixed", opt="cg", scf=True,
          monitor=True, steps=40),
        # the test suite's small system with a fixed V(r) and every option at its default
        m(name="water8-fp64-fixed", nmol=8, ecut=30.0, grid=48, precision="fp64", opt="sd",
          scf=False, resid=True, monitor=True, steps=40),
        # the benchmark's system and options, both precisions
        m(name="water32-mixed", nmol=32, ecut=70.0, precision="mixed", opt="sd", scf=True,
          autotune=True, steps=100),
        m(name="water32-fp64", nmol=32, ecut=70.0, precision="fp64", opt="sd", scf=True,
          autotune=True, steps=80),
        # ragged state count, with the non-local projectors
        m(name="water21-fp64-kb-cg", nmol=21, ecut=60.0, precision="fp64", opt="cg", scf=True,
          nonlocal_kb=True, monitor=True, steps=30),
        # a cell with three different sides, so the planes are not square
        m(name="water24-mixed-brick", nmol=24, ecut=50.0, shape="brick", precision="mixed",
          opt="sd", scf=True, steps=40),
        # the largest requests of the request loop, a ragged and a full one
        m(name="water45-mixed-cg", nmol=45, ecut=60.0, precision="mixed", opt="cg", scf=True,
          steps=32),
        m(name="water64-fp64-cg", nmol=64, ecut=70.0, precision="fp64", opt="cg", scf=True,
          steps=24),
        # the largest system
        m(name="water128-mixed", nmol=128, ecut=70.0, precision="mixed", opt="sd", scf=True,
          steps=32),
        # the request loop: six sizes at once, half of them in mixed precision
        dict(name="serve-6", kind="serve", first=4, last=36, count=6, ecut=60.0, steps=25),
    ]


def draw(rng):
    kind = rng.choices(("minimise", "ortho", "serve"), (8, 1, 1))[0]
    if kind == "ortho":
        return dict(kind=kind, n=int(round(math.exp(rng.uniform(math.log(17), math.log(400))))))
    ecut = rng.choice((30.0, 50.0, 60.0, 70.0))
    if kind == "serve":
        return dict(kind=kind, first=rng.randint(4, 8), last=rng.randint(12, 40),
                    count=rng.randint(3, 6), ecut=max(50.0, ecut), steps=rng.randint(15, 25))
    nmol = int(round(math.exp(rng.uniform(math.log(4), math.log(64)))))
    opt = rng.choice(("sd", "cg"))
    return dict(kind=kind, nmol=nmol, ecut=ecut, shape=rng.choice(("cubic", "cubic", "cubic", "brick")),
                precision=rng.choice(("fp64", "mixed")), opt=opt,
                scf=rng.choice((True, True, False)),
                nonlocal_kb=rng.random() < 0.3, resid=rng.random() < 0.3,
                monitor=rng.random() < 0.5, autotune=rng.random() < 0.2,
                steps=rng.randint(8, max(9, min(40, 800 // nmol))))


# ------------------------------------------------------------------ inputs


def _sides(nmol, shape):
    """Box sides (A) at the density of 32 molecules in 9.86 A."""
    a = 9.86 * (nmol / 32.0) ** (1.0 / 3.0)
    return (a, a, a) if shape == "cubic" else (0.85 * a, a, a / 0.85)


def _grid(case):
    """The case's own cubic grid, or the smallest compiled lengths that hold
    |G|^2 <= 4 ecut on every axis."""
    if "grid" in case:
        return (case["grid"],) * 3
    sides, ecut = _sides(case["nmol"], case.get("shape", "cubic")), case["ecut"]
    need = [2 * int(2.0 * math.sqrt(ecut) * s * BOHR / (2.0 * math.pi) + PAD) + 1 for s in sides]
    return tuple(next(n for n in system.FFT_SIZES if n >= k) for k in need)


def _liquid(nmol, sides, rng):
    """Molecules at random, oxygens at least 2.5 A apart, random orientations:
    positions in bohr and species 0 (O) or 1 (H)."""
    box = np.asarray(sides)
    oxy = np.zeros((0, 3))
    while len(oxy) < nmol:
        p = rng.uniform(0.0, 1.0, 3) * box
        d = oxy - p
        d -= box * np.round(d / box)
        if len(oxy) == 0 or (d * d).sum(axis=1).min() >= 2.5 ** 2:
            oxy = np.concatenate([oxy, p[None]])
    half = math.radians(system.HOH_DEG) / 2.0
    arms = system.OH_ANG * np.array([[math.sin(half), math.cos(half), 0.0],
                                     [-math.sin(half), math.cos(half), 0.0]])
    pos, species = [], []
    for o in oxy:
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        pos += [o, o + q @ arms[0], o + q @ arms[1]]
        species += [0, 1, 1]
    return np.mod(np.array(pos), box) * BOHR, np.array(species, np.int32)


def _orthonormal(kx, g2, nstates, seed):
    """Gaussian-weighted random coefficients, real in r, orthonormal with
    norm 2 under the weights 1 (kx = 0) and 2: [nstates][npts] complex."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    npts = len(kx)
    nkx0 = int((kx == 0).sum())
    amp = torch.exp(torch.from_numpy(g2).cuda() / -4.0)
    c = torch.randn(nstates, npts, 2, generator=gen, device="cuda", dtype=torch.float64)
    c *= amp[None, :, None]
    # the stored kx = 0 points are symmetric about G = 0: the first half is
    # the mirror of the second
    mid = nkx0 // 2
    c[:, mid, 1] = 0.0
    mirror = c[:, mid + 1:nkx0].flip(1)
    c[:, :mid, 0] = mirror[..., 0]
    c[:, :mid, 1] = -mirror[..., 1]
    w = torch.full((npts,), math.sqrt(2.0), device="cuda", dtype=torch.float64)
    w[:nkx0] = 1.0
    for _ in range(2):
        a = (c * w[None, :, None]).reshape(nstates, -1)
        low = torch.linalg.cholesky((a @ a.T).cpu())
        inv = torch.linalg.solve_triangular(low, torch.eye(nstates, dtype=torch.float64),
                                            upper=False).cuda()
        c = (inv @ c.reshape(nstates, -1)).reshape(nstates, npts, 2)
    return torch.view_as_complex((c * math.sqrt(2.0)).contiguous())


def _system(case, seed):
    """Everything a program holds before it makes a context."""
    sides = _sides(case["nmol"], case.get("shape", "cubic"))
    ecut = float(case["ecut"])
    grid = _grid(case)
    hmat = np.diag([s * BOHR for s in sides]).reshape(9)
    rng = np.random.Generator(np.random.PCG64([int(seed), 17]))
    pos, species = _liquid(case["nmol"], sides, rng)
    kx, ky, kz = _lib.kvecs(ecut, hmat)
    g2 = system.gvec_sq(kx, ky, kz, hmat)
    nstates = 4 * case["nmol"]
    psi = _orthonormal(kx, g2, nstates, int(seed) % (1 << 62))
    params = {"O": (float(rng.uniform(-6.5, -5.5)), float(rng.uniform(0.95, 1.05))),
              "H": (float(rng.uniform(-1.3, -1.1)), float(rng.uniform(0.55, 0.65)))}
    s = dict(hmat=hmat, grid=grid, ecut_ry=ecut, nstates=nstates, kx=kx, ky=ky, kz=kz, g2=g2,
             pos=pos, species=species, pseudo=system.local_pseudo_tables(params, ecut),
             psi=psi.cpu().numpy())
    if case.get("nonlocal_kb"):
        t = system.nonlocal_tables(system.kb_params(int(seed) % (1 << 31)), ecut)
        ox = pos[species == 0]
        s["kb"] = dict(pos=ox, species=np.zeros(len(ox), np.int32), gmin=t["gmin"], dg=t["dg"],
                       proj=t["proj"], proj_g0=t["proj_g0"], vnorm=t["vnorm"])
    if case["kind"] == "minimise" and not case["scf"]:
        s["vks"] = _fixed_potential(pos, species, params, sides, grid)
    return s


def _fixed_potential(pos, species, params, sides, grid):
    """Gaussian wells at the atoms, nearest image: V[z][y][x] (Ha)."""
    v = torch.zeros(grid[2], grid[1], grid[0], dtype=torch.float64, device="cuda")
    for sp, name in enumerate(("O", "H")):
        a, sig = params[name]
        e = []
        for d in range(3):
            side = sides[d] * BOHR
            x = np.arange(grid[d])[None, :] * (side / grid[d]) - pos[species == sp][:, d, None]
            x -= side * np.round(x / side)
            e.append(torch.from_numpy(np.exp(-x * x / (2.0 * sig * sig))).cuda())
        v += a * torch.einsum("az,ay,ax->zyx", e[2], e[1], e[0])
    return v.cpu().numpy()


def _requests(case):
    """The requests of one serve case: sizes spread geometrically, every
    other one in mixed precision."""
    out = []
    for i in range(case["count"]):
        r = case["first"] * (case["last"] / case["first"]) ** (i / (case["count"] - 1))
        out.append(dict(kind="minimise", nmol=int(round(r)), ecut=case["ecut"], scf=True, opt="cg",
                        precision="mixed" if i % 2 else "fp64", steps=case["steps"]))
    return out


def _matrix(case, seed):
    """S of a set of norm-2 states after an update that moved them a little."""
    rng = np.random.Generator(np.random.PCG64([int(seed), 23]))
    n = case["n"]
    e = rng.normal(size=(n, n)) * (0.05 / math.sqrt(n))
    return 2.0 * np.eye(n) + e + e.T


# ------------------------------------------------------------------ the calls


def prepare(case, seed):
    if case["kind"] == "ortho":
        return dict(case=case, S=_matrix(case, seed))
    if case["kind"] == "serve":
        reqs = _requests(case)
        return dict(case=case, reqs=reqs,
                    systems=[_system(r, seed * 64 + i) for i, r in enumerate(reqs)],
                    server=serve.Server(max_active=8))
    s = _system(case, seed)
    c = CPContext(s["grid"], s["hmat"], s["ecut_ry"], s["nstates"], s["kx"], s["ky"], s["kz"],
                  precision=case["precision"], dt=DT[case["opt"]],
                  ns_tol=1e-15 if case["precision"] == "fp64" else 1e-14,
                  want_resid=int(case["resid"]), use_cg=int(case["opt"] == "cg"),
                  vks_from_rho=int(case["scf"]), autotune=int(case["autotune"]))
    t = s["pseudo"]
    if case["scf"]:
        c.set_local_pseudo(s["pos"], s["species"], t["gmin"], t["dg"], t["vps"], t["vps_g0"])
    else:
        c.set_vks(s["vks"])
    if "kb" in s:
        c.set_nonlocal(**s["kb"])
    return dict(case=case, ctx=c, psi=s["psi"])


def _result(precision, energies, psi):
    psi = torch.from_numpy(psi)
    if precision == "mixed":
        return dict(energies=np.asarray(energies, np.float32), psi=psi.to(torch.complex64))
    return dict(energies=np.asarray(energies, np.float64), psi=psi)


def run(state):
    case = state["case"]
    if case["kind"] == "ortho":
        return _lib.ortho_transform(state["S"])[0]
    if case["kind"] == "serve":
        srv = state["server"]
        for i, (r, s) in enumerate(zip(state["reqs"], state["systems"])):
            srv.submit(s, i, f_tol=1e-12, max_steps=r["steps"], precision=r["precision"],
                       want_psi=True, scf=True, fp64_below=0.0, dt=DT["cg"], use_cg=1, ns_mode=6,
                       want_resid=0)
        got = {r["tag"]: r for r in srv.drain()}
        return [_result(r["precision"], [got[i]["eelec"], got[i]["fnorm"]], got[i]["psi"])
                for i, r in enumerate(state["reqs"])]
    c = state["ctx"]
    c.set_psi(state["psi"])
    for _ in range(case["steps"] - 1):
        c.step(fetch=case["monitor"])
    r = c.step()
    return _result(case["precision"], [r[k] for k in ENERGIES], c.get_psi())


ENERGIES = ("eke", "eloc", "ehart", "exc", "enl", "eelec", "fnorm")


# ------------------------------------------------------------------ its work


def work(case):
    """Per step: the pruned transforms' and the four products' operations;
    the coefficients read and written, the forces written, rho and V."""
    if case["kind"] == "ortho":
        n = case["n"]
        return dict(bytes=2 * 8 * n * n, flops=5 * 6 * n ** 3)
    if case["kind"] == "serve":
        w = [work(r) for r in _requests(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    sides = _sides(case["nmol"], case.get("shape", "cubic"))
    ecut, n = case["ecut"], 4 * case["nmol"]
    grid = _grid(case)
    points = float(np.prod(grid))
    volume = float(np.prod(sides)) * BOHR ** 3
    npts = volume * ecut ** 1.5 / (6.0 * math.pi ** 2) / 2.0  # half sphere
    # real transforms, 2.5 N log2 N each, about half of it on populated lines
    fft = 2 * n * 2.5 * points * math.log2(points) / 2
    products = 2.0 * n * n * (2 * npts) * 3.5  # Lambda, its projection, Psi T, half of S
    per = dict(bytes=3 * 16.0 * n * npts + 2 * 8 * points, flops=fft + products)
    if case.get("nonlocal_kb"):
        per["flops"] += 2 * 2.0 * n * case["nmol"] * 2 * npts
    return {k: v * case["steps"] for k, v in per.items()}


# ------------------------------------------------------------------ the same in 64 bits


def _gvectors(grid, hmat):
    """Half-space (kx >= 0) frequencies of a real transform: G components,
    [nz][ny][nx/2+1], and the weights 1 (kx = 0) and 2."""
    hi = np.linalg.inv(np.asarray(hmat).reshape(3, 3))
    f = [torch.from_numpy(np.fft.fftfreq(n, 1.0 / n)).cuda() for n in grid]
    f[0] = torch.arange(grid[0] // 2 + 1, dtype=torch.float64, device="cuda")
    k = (f[0][None, None, :], f[1][None, :, None], f[2][:, None, None])
    shape = (grid[2], grid[1], grid[0] // 2 + 1)
    g = [2.0 * math.pi * sum(hi[r, a] * k[a] for a in range(3)).expand(shape) for r in range(3)]
    w = torch.where(k[0] == 0, 1.0, 2.0).expand(shape)
    return g, w


def _spline(tab, gmin, dg, g):
    """Rows c0..c3 on a uniform grid at the points g."""
    tab = torch.from_numpy(np.ascontiguousarray(tab)).cuda()
    i = torch.clamp(((g - gmin) / dg + 1.0).long(), 1, tab.shape[1]) - 1
    h = g - (i.double() * dg + gmin)
    return ((tab[3][i] * h + tab[2][i]) * h + tab[1][i]) * h + tab[0][i]


def _form(tab, at_zero, t, g):
    return torch.where(g > 0, _spline(tab, t["gmin"], t["dg"], g), torch.as_tensor(at_zero, device="cuda"))


def _local_potential(s, g, inside):
    """(1/Omega) sum_I v_I(|G|) exp(-i G.R_I) on the points `inside`."""
    t = s["pseudo"]
    gi = torch.stack([x[inside] for x in g])
    mod = torch.sqrt((gi * gi).sum(0))
    out = torch.zeros(gi.shape[1], dtype=torch.complex128, device="cuda")
    for sp in range(2):
        sf = torch.zeros_like(out)
        for r in torch.from_numpy(s["pos"][s["species"] == sp]).cuda():
            sf += torch.exp(-1j * (r[:, None] * gi).sum(0))
        out += sf * _form(t["vps"][sp], t["vps_g0"][sp], t, mod)
    return out / abs(np.linalg.det(s["hmat"].reshape(3, 3)))


def _exchange_correlation(rho):
    """Perdew-Zunger LDA: (eps_x, eps_c, their potential) per electron."""
    rs = (3.0 / (4.0 * math.pi * rho)) ** (1.0 / 3.0)
    sq, lg = torch.sqrt(rs), torch.log(rs)
    vx = -(3.0 * rho / math.pi) ** (1.0 / 3.0)
    low = -0.1423 / (1.0 + 1.0529 * sq + 0.3334 * rs)
    vlow = low * (1.0 + 7.0 / 6.0 * 1.0529 * sq + 4.0 / 3.0 * 0.3334 * rs) / (1.0 + 1.0529 * sq + 0.3334 * rs)
    high = 0.0311 * lg - 0.048 + 0.002 * rs * lg - 0.0116 * rs
    vhigh = 0.0311 * lg + (-0.048 - 0.0311 / 3.0) + 2.0 / 3.0 * 0.002 * rs * lg + (2.0 * -0.0116 - 0.002) / 3.0 * rs
    return 0.75 * vx, torch.where(rs >= 1.0, low, high), vx + torch.where(rs >= 1.0, vlow, vhigh)


def _minimise(case, s):
    """`steps` steps in plain torch, FP64: the last step's energies and the
    coefficients after it."""
    grid, n = s["grid"], s["nstates"]
    nx, ny, nz = grid
    total = nx * ny * nz
    volume = abs(np.linalg.det(s["hmat"].reshape(3, 3)))
    cell = volume / total
    kx = torch.from_numpy(s["kx"].astype(np.int64)).cuda()
    flat = torch.from_numpy((s["kz"].astype(np.int64) % nz * ny + s["ky"] % ny) * (nx // 2 + 1) + s["kx"]).cuda()
    nkx0 = int((kx == 0).sum())
    mid = nkx0 // 2
    w = torch.where(kx == 0, 1.0, 2.0).double()
    g2 = torch.from_numpy(s["g2"]).cuda()
    # fictitious masses: CP_create_mass with tau = 25 fs and the 2 Ry cutoff
    m0 = 2.0 * (25.0 / 0.0241888) ** 2 * 0.00050
    dtm = DT[case["opt"]] / torch.where(g2 > 2.0, w * g2 * (m0 / 2.0), w * m0)
    psi = torch.from_numpy(s["psi"]).cuda()
    batch = max(1, int(2e7 // total))
    if case["scf"]:
        g, wg = _gvectors(grid, s["hmat"])
        gg = g[0] ** 2 + g[1] ** 2 + g[2] ** 2
        inside = gg <= 4.0 * s["ecut_ry"]
        vloc = _local_potential(s, g, inside)
        gs, ws = gg[inside], wg[inside]
        coul = torch.where(gs > 0, 4.0 * math.pi / (torch.where(gs > 0, gs, 1.0) * volume), 0.0)
    else:
        v = torch.from_numpy(s["vks"]).cuda()
    if "kb" in s:
        t = s["kb"]
        hi = torch.from_numpy(np.linalg.inv(s["hmat"].reshape(3, 3))).cuda()
        k = torch.stack([kx, torch.from_numpy(s["ky"].astype(np.int64)).cuda(),
                         torch.from_numpy(s["kz"].astype(np.int64)).cuda()]).double()
        gv = 2.0 * math.pi * (hi @ k)
        phase = (torch.from_numpy(t["pos"]).cuda()[:, :, None] * gv[None]).sum(1)
        proj = _form(t["proj"][0], t["proj_g0"][0], t, torch.sqrt(g2)) / math.sqrt(4.0 * math.pi)
        sf = proj * torch.exp(-1j * phase)
        vn = float(t["vnorm"][0]) / volume

    def real_dot(a, b):
        return torch.view_as_real(a).reshape(len(a), -1) @ torch.view_as_real(b).reshape(len(b), -1).T

    def mix(m, a):  # sum_i m[i][j] a[i]
        return torch.view_as_complex((m.T @ torch.view_as_real(a).reshape(len(a), -1)).reshape(m.shape[1], -1, 2).contiguous())

    def real_space(a):
        half = torch.zeros(len(a), nz * ny * (nx // 2 + 1), dtype=torch.complex128, device="cuda")
        half[:, flat] = a.conj()
        return torch.fft.irfftn(half.reshape(len(a), nz, ny, nx // 2 + 1), s=(nz, ny, nx), norm="forward")

    direction, old, since = torch.zeros_like(psi), None, 0
    for _ in range(case["steps"]):
        rho = torch.zeros(nz, ny, nx, dtype=torch.float64, device="cuda")
        for i in range(0, n, batch):
            rho += (real_space(psi[i:i + batch]) ** 2).sum(0)
        rho /= volume
        ehart = exc = enl = 0.0
        if case["scf"]:
            ex, ec, vxc = _exchange_correlation(rho)
            rg = torch.fft.rfftn(rho * cell)[inside]
            ehart = float((0.5 * coul * ws * (rg.real ** 2 + rg.imag ** 2)).sum())
            eloc = float((ws * (rg.real * vloc.real + rg.imag * vloc.imag)).sum())
            exc = float(((ex + ec) * rho).sum()) * cell
            vg = torch.zeros(nz, ny, nx // 2 + 1, dtype=torch.complex128, device="cuda")
            vg[inside] = coul * rg + vloc
            v = vxc + torch.fft.irfftn(vg, s=(nz, ny, nx), norm="forward")
        else:
            eloc = float((v * rho).sum()) * cell
        force = torch.empty_like(psi)
        for i in range(0, n, batch):
            u = torch.fft.rfftn(real_space(psi[i:i + batch]) * v, dim=(1, 2, 3)).reshape(-1, nz * ny * (nx // 2 + 1))
            force[i:i + batch] = u[:, flat].conj() * (w * (-2.0 / total)) - (w * g2) * psi[i:i + batch]
        eke = 0.5 * float((w * g2 * (psi.real ** 2 + psi.imag ** 2)).sum())
        if "kb" in s:
            z = real_dot(psi * w, sf)
            enl = vn * float((z * z).sum())
            force -= w * mix(2.0 * vn * z.T.contiguous(), sf)
        force -= torch.where(kx == 0, 0.5, 1.0) * mix(real_dot(psi, force), psi)
        f2 = float((force.real ** 2 + force.imag ** 2).sum())
        if case["opt"] == "cg":
            fnorm = math.sqrt(f2)
            reset = old is None or (fnorm > 1.05 * old and since >= 5) or fnorm > 2.0 * old
            gamma = 0.0 if reset else (fnorm / old) ** 2
            since = 1 if reset else since + 1
            old = fnorm
            direction = direction * gamma + force
        else:
            direction = force
        psi = psi + dtm * direction
        psi[:, :mid] = psi[:, mid + 1:nkx0].flip(1).conj()
        e, q = torch.linalg.eigh((real_dot(psi * w, psi) / 2.0).cpu())
        psi = mix(((q / torch.sqrt(e)) @ q.T).cuda(), psi)
    eelec = eke + eloc + ehart + exc + enl
    return [eke, eloc, ehart, exc, enl, eelec, math.sqrt(f2)], psi


def exact(case, seed):
    if case["kind"] == "ortho":
        e, q = np.linalg.eigh(_matrix(case, seed) / 2.0)
        return (q / np.sqrt(e)) @ q.T
    if case["kind"] == "serve":
        out = []
        for i, r in enumerate(_requests(case)):
            e, psi = _minimise(r, _system(r, seed * 64 + i))
            out.append(dict(energies=np.array([e[5], e[6]]), psi=psi))
        return out
    e, psi = _minimise(case, _system(case, seed))
    return dict(energies=np.array(e), psi=psi)
