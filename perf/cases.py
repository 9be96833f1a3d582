"""Performance cases of the PMG solver, through its public entry points.

A case is a dict of plain values.  `listed()` holds the fixed ones, `draw()`
gives another of the same ranges, `prepare()` makes what a program has in
hand before the call (resident contexts, a running server, host arrays of
the drop-in driver), `run()` is one pass as such a program makes it, `work()`
the bytes and operations that pass cannot do without and `exact()` the
result in 64 bits from plain torch.

Kinds of pass:
  request   another molecule into a resident context (GPU assembly, operator
            build), the linear solve to 1e-6, the potential to the host
  newton    the same with the nonlinear (sinh) term, Newton to 1e-8
  pcg       the same with the class-style preconditioned CG
  dropin    the reference-shaped driver call on host arrays
  serve     a batch of requests of uneven sizes to a running server
  residual  the allocation-free FP64 residual on caller-owned device arrays
"""
import math

import numpy as np
import torch

import multigrid_amd as mg

MODES = {"fp64": mg.PMG_FP64, "mixed": mg.PMG_MIXED}
IONS = ([1.0, -1.0], [0.5, 0.5])  # 1:1 salt of the nonlinear term
SERVE_SIZES = (65, 97, 129, 161)


def listed():
    return [
        # the smallest grid of the serving table: launches and host round
        # trips, hardly any data
        dict(name="request33_mixed", kind="request", mode="mixed", n=33, nlev=3, h=0.5,
             natoms=40, radius=6.0, ionic=0.15, charges=0),
        # the 65^3 benchmark workload in the drop-in's precision
        dict(name="request65_fp64", kind="request", mode="fp64", n=65, nlev=4, h=0.5,
             natoms=200, radius=14.0, ionic=0.15, charges=0),
        # a middle request of the serving stream, its rows not a multiple of
        # any tile
        dict(name="request97_mixed", kind="request", mode="mixed", n=97, nlev=5, h=0.5,
             natoms=600, radius=16.0, ionic=0.15, charges=0),
        # the 161^3 benchmark workload, both precisions
        dict(name="solve161_mixed", kind="request", mode="mixed", n=161, nlev=5, h=0.4,
             natoms=1000, radius=25.0, ionic=0.15, charges=0),
        dict(name="solve161_fp64", kind="request", mode="fp64", n=161, nlev=5, h=0.4,
             natoms=1000, radius=25.0, ionic=0.15, charges=0),
        # the large single solve of the benchmark
        dict(name="solve289_mixed", kind="request", mode="mixed", n=289, nlev=6, h=0.35,
             natoms=5000, radius=45.0, ionic=0.15, charges=1),
        # the nonlinear solve: a small one in FP64 and the 129^3 benchmark
        # workload with FP32 inner cycles
        dict(name="newton65_fp64", kind="newton", mode="fp64", n=65, nlev=4, h=0.5,
             natoms=200, radius=14.0, ionic=0.15, charges=0),
        dict(name="newton129_mixed", kind="newton", mode="mixed", n=129, nlev=5, h=0.5,
             natoms=800, radius=20.0, ionic=0.30, charges=0),
        # the class-style solver on the 161^3 workload
        dict(name="pcg161_fp64", kind="pcg", mode="fp64", n=161, nlev=5, h=0.4,
             natoms=1000, radius=25.0, ionic=0.15, charges=0),
        # one call of the reference-shaped driver on a box with three
        # different sides: allocation, copies, build, solve, work arrays back
        dict(name="dropin_ragged", kind="dropin", mode="fp64", nx=65, ny=97, nz=81, nlev=5,
             h=0.5, natoms=200, radius=12.0, ionic=0.15, charges=0),
        # a batch of the serving stream, eight solves in flight
        dict(name="serve16_mixed", kind="serve", mode="mixed", requests=16, active=8, groups=0,
             h=0.5, ionic=0.15, atoms_low=100, atoms_high=3000),
        # the outer residual of a caller's own loop on the device
        dict(name="residual161", kind="residual", nx=161, ny=161, nz=161),
    ]


# Grid sizes n = (c - 1) 2^(levels-1) + 1 with a coarsest side c of 5 to 11.
SIZES = {33: 3, 41: 3, 49: 4, 65: 4, 81: 4, 97: 5, 113: 5, 129: 5, 145: 5, 161: 5, 193: 6,
         225: 6, 257: 6, 289: 6}


def _fit(n, h, natoms):
    """Radius of a ball of natoms at the density of the 65^3 workload that
    leaves room in an n^3 box."""
    return min(14.0 * (natoms / 200.0) ** (1.0 / 3.0), 0.75 * (n - 1) * h / 2 - 2.0)


def draw(rng):
    kind = rng.choices(("request", "newton", "pcg", "dropin", "serve", "residual"),
                       (8, 2, 2, 2, 2, 2))[0]

    def size(most, least=33):
        t = math.exp(rng.uniform(math.log(least), math.log(most + 8)))
        return min((n for n in SIZES if least <= n <= most), key=lambda n: abs(n - t))

    if kind == "residual":
        return dict(kind=kind, nx=rng.randint(20, 289), ny=rng.randint(20, 200),
                    nz=rng.randint(20, 200))
    if kind == "serve":
        mode = rng.choice(("mixed", "fp64"))
        return dict(kind=kind, mode=mode, requests=rng.randint(5, 14 if mode == "mixed" else 10),
                    active=rng.choice((4, 8)), groups=rng.choice((0, 0, 2)), h=0.5, ionic=0.15,
                    atoms_low=100, atoms_high=rng.randint(500, 3000))
    h, ionic = round(rng.uniform(0.3, 0.6), 3), rng.choice((0.05, 0.15, 0.30))
    if kind == "dropin":
        nlev = rng.choice((4, 5))
        low = 4 if nlev == 4 else 3
        nx, ny, nz = ((rng.randint(low, 7) << (nlev - 1)) + 1 for _ in range(3))
        natoms = int(math.exp(rng.uniform(math.log(50), math.log(400))))
        return dict(kind=kind, mode="fp64", nx=nx, ny=ny, nz=nz, nlev=nlev, h=h, natoms=natoms,
                    radius=_fit(min(nx, ny, nz), h, natoms), ionic=ionic, charges=0)
    mode = rng.choice(("mixed", "mixed", "fp64"))
    n = size({"request": 289 if mode == "mixed" else 193, "newton": 129, "pcg": 161}[kind])
    most = min(5000, 200 * (n / 65.0) ** 3 * 2)
    natoms = int(math.exp(rng.uniform(math.log(40), math.log(most))))
    return dict(kind=kind, mode=mode, n=n, nlev=SIZES[n], h=h, natoms=natoms,
                radius=_fit(n, h, natoms), ionic=ionic, charges=rng.choice((0, 1)))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _molecule(natoms, radius, charges, seed):
    """natoms x {x, y, z, radius, charge}: atoms uniform in a ball, radii
    1.2 to 2.0 A, charges +-1 (net zero, one left over is 0) or one of
    {-1, -0.5, 0, 0.5, 1}."""
    g = np.random.default_rng(seed)
    v = g.standard_normal((natoms, 3))
    v *= (radius * g.random(natoms) ** (1.0 / 3.0) / np.linalg.norm(v, axis=1))[:, None]
    if charges:
        q = g.choice([-1.0, -0.5, 0.0, 0.5, 1.0], natoms)
    else:
        q = np.where(np.arange(natoms) % 2 == 0, 1.0, -1.0)
        if natoms % 2:
            q[-1] = 0.0
    return np.ascontiguousarray(np.column_stack([v, g.uniform(1.2, 2.0, natoms), q]))


def _requests(case, seed):
    """(n, levels, atoms) of the requests of a batch: the sizes in turn, so
    that every batch holds each of them."""
    g = np.random.default_rng([seed, 1])
    out = []
    for q in range(case["requests"]):
        n = SERVE_SIZES[q % len(SERVE_SIZES)]
        natoms = int(g.integers(case["atoms_low"], case["atoms_high"] + 1))
        out.append((n, mg.SERVE_LEVELS[n],
                    _molecule(natoms, _fit(n, case["h"], natoms), 0, int(g.integers(1 << 40)))))
    return out


def _params(nx, ny, nz, nlev, **kw):
    sz = mg.Vmgsz(2, 0, 0, nx, ny, nz, nlev)
    return mg.Vpackmg(sz["iretot"], sz["iintot"], nx, ny, nz, nlev, **kw) + (sz,)


def _pick(mask, a, b):
    """a where mask holds, else b, in 64 bits."""
    like = torch.zeros((), device=mask.device, dtype=torch.float64)
    return torch.where(mask, like + a, like + b)


def _residual_inputs(case, seed, device):
    """A 7-point operator with a dielectric step (couplings of 2 to 78.5),
    a right-hand side and an iterate, as flat device arrays."""
    g = torch.Generator(device=device).manual_seed(seed)
    shape = (case["nz"], case["ny"], case["nx"])

    def rand(*s):
        return torch.rand(*s, generator=g, device=device, dtype=torch.float64)

    eps = _pick(rand(*shape) < 0.3, 2.0, 78.54)
    ac = torch.zeros((4,) + shape, device=device, dtype=torch.float64)
    for p, d in ((1, 2), (2, 1), (3, 0)):  # oE, oN, uC: faces towards i+1, j+1, k+1
        up = torch.roll(eps, -1, d)
        ac[p] = 2 * eps * up / (eps + up) * 0.4
        for q in (0, shape[d] - 2, shape[d] - 1):  # couplings to the boundary are folded away
            ac[p].select(d, q).zero_()
        ac[0] += ac[p] + torch.roll(ac[p], 1, d)
    ac[0] += 0.1
    cc = _pick(rand(*shape) < 0.5, 0.0, 0.05)
    fc = rand(*shape) - 0.5
    x = 3.0 * (rand(*shape) - 0.5)
    return ac, cc, fc, x


def prepare(case, seed):
    kind = case["kind"]
    if kind == "residual":
        ac, cc, fc, x = _residual_inputs(case, seed, "cuda")
        for a, planes in ((ac, 4), (cc, 1), (fc, 1), (x, 1)):  # raw pointers follow
            assert a.dtype == torch.float64 and a.is_contiguous()
            assert a.numel() == planes * case["nx"] * case["ny"] * case["nz"]
        return dict(kind=kind, dims=(case["nx"], case["ny"], case["nz"]), arrays=(ac, cc, fc, x),
                    r=torch.zeros(x.shape, device="cuda", dtype=torch.float32),
                    l1=torch.zeros(1, device="cuda", dtype=torch.float64))
    if kind == "serve":
        reqs = _requests(case, seed)
        srv = mg.Server(64 << 30, case["active"], groups=case["groups"])
        par = {n: mg.make_params(n, nlev) for n, nlev, _ in reqs}
        state = dict(kind=kind, srv=srv, par=par, mode=MODES[case["mode"]], h=case["h"],
                     ionic=case["ionic"], reqs=[(n, a) for n, _, a in reqs])
        # a running service holds a context of every shape and precision
        small = _molecule(100, 8.0, 0, seed)
        for t in [srv.submit(*par[n], state["mode"], case["h"], case["ionic"], small,
                             want_u=False) for n, _, _ in reqs]:
            srv.wait(t)
        return state
    atoms = _molecule(case["natoms"], case["radius"], case["charges"], seed)
    if kind == "dropin":
        dims = case["nx"], case["ny"], case["nz"]
        inp = _assemble(dims, case["h"], case["ionic"], atoms, "cuda")
        iparm, rparm, sz = _params(*dims, case["nlev"])
        return dict(kind=kind, args=(iparm, rparm), iwork=np.zeros(sz["iintot"], np.int32),
                    rwork=np.zeros(sz["iretot"]), u=np.zeros(dims[0] * dims[1] * dims[2]),
                    arrays=_driver_arrays(inp))
    n = case["n"]
    if kind == "newton":
        mg.Vmypdefinitnpbe(2, *IONS)
        iparm, rparm = mg.make_params(n, case["nlev"], nonlin=1, errtol=1e-8)
    else:
        iparm, rparm = mg.make_params(n, case["nlev"])
    mol = (case["h"], case["ionic"], atoms)
    return dict(kind=kind, ctx=mg.Context(iparm, rparm, pbe=mol), mol=mol,
                mode=MODES[case["mode"]])


def run(state):
    kind = state["kind"]
    if kind == "residual":
        ac, cc, fc, x = state["arrays"]
        rc = mg.lib().pmg_mresid_mixed_noalloc(
            *state["dims"], ac.data_ptr(), cc.data_ptr(), fc.data_ptr(), x.data_ptr(),
            state["r"].data_ptr(), state["l1"].data_ptr(),
            torch.cuda.current_stream().cuda_stream)
        if rc:
            raise mg.PMGError(rc, "residual")
        return {"r": state["r"], "l1": state["l1"]}
    if kind == "serve":
        srv = state["srv"]
        got = [srv.wait(t) for t in
               [srv.submit(*state["par"][n], state["mode"], state["h"], state["ionic"], atoms)
                for n, atoms in state["reqs"]]]
        return {"u": [g["u"] for g in got], "iters": [g["iters"] for g in got]}
    if kind == "dropin":
        mg.Vmgdriv(*state["args"], state["iwork"], state["rwork"], state["u"], *state["arrays"])
        return {"u": state["u"], "rwork": state["rwork"], "iters": mg.last_stats()[0]}
    ctx = state["ctx"]
    ctx.load_pbe(*state["mol"])
    if kind == "pcg":
        ctx.pcg(state["mode"])
    else:
        ctx.solve(state["mode"])
    return {"u": ctx.u(), "iters": ctx.stats()["iters"]}


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
def _solve_work(nx, ny, nz, nlev, mode, cycles, natoms):
    """Bytes and operations of a solve of `cycles` V(2,2) cycles: on each
    level the operator, the right-hand side and the iterate pass once on the
    way down and once on the way up, the prolongation likewise; the mixed
    solve's outer residual reads the FP64 operator once per cycle.  The
    build writes the hierarchy once."""
    w = 4 if mode == "mixed" else 8
    cyc = build = flops = 0.0
    dims = nx, ny, nz
    for lev in range(nlev):
        p = float(dims[0] * dims[1] * dims[2])
        if lev == 0:
            cyc += p * w * (6 + 7)
            cyc += p * (8 * 7 if mode == "mixed" else 8 * 6)
            build += p * 8 * (5 + 7)
            flops += p * 6 * 14
        else:
            cyc += p * w * (16 + 17) + p * w * 27 * 2
            build += p * (8 + (w if w == 4 else 0)) * (14 + 27 + 2)
            flops += p * (6 * 54 + 2 * 54)
        dims = tuple((d - 1) // 2 + 1 for d in dims)
    faces = 2.0 * (nx * ny + ny * nz + nx * nz) * natoms
    return {"bytes": build + cycles * cyc + 8.0 * nx * ny * nz,
            "flops": cycles * flops + 40 * faces}


def work(case):
    kind = case["kind"]
    if kind == "residual":
        n = case["nx"] * case["ny"] * case["nz"]
        return {"bytes": n * (7 * 8 + 4), "flops": n * 16}
    if kind == "serve":
        mid = (case["atoms_low"] + case["atoms_high"]) // 2
        parts = [_solve_work(n, n, n, mg.SERVE_LEVELS[n], case["mode"], 8, mid)
                 for n in (SERVE_SIZES[q % len(SERVE_SIZES)] for q in range(case["requests"]))]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "dropin":
        w = _solve_work(case["nx"], case["ny"], case["nz"], case["nlev"], "fp64", 8,
                        case["natoms"])
        w["bytes"] += 8.0 * mg.Vmgsz(2, 0, 0, case["nx"], case["ny"], case["nz"],
                                     case["nlev"])["iretot"]
        return w
    cycles = {"request": 8, "newton": 16, "pcg": 7}[kind]
    return _solve_work(case["n"], case["n"], case["n"], case["nlev"], case["mode"], cycles,
                       case["natoms"])


# ---------------------------------------------------------------------------
# The grid problem in plain torch
# ---------------------------------------------------------------------------
def _constants(ionic):
    kb, qe, eps0, na, temp = 1.380649e-23, 1.602176634e-19, 8.8541878128e-12, 6.02214076e23, 298.15
    bjerrum = qe * qe / (4.0 * math.pi * eps0 * kb * temp) * 1e10
    kap2 = 2.0 * ionic * 1000.0 * na * qe * qe / (eps0 * 78.54 * kb * temp) * 1e-20
    return bjerrum, kap2


def _assemble(dims, h, ionic, atoms, device):
    """The grid inputs of a molecule centred in an nx x ny x nz box of
    spacing h, as 64-bit tensors indexed [k, j, i]: face coefficients a1-a3
    (2 inside the atom spheres, 78.54 outside, harmonic averages), the ion
    term cc (0 within 2 A of an atom), the charge source, and the boundary
    values u (Debye-Hueckel spheres; 0 inside)."""
    f64 = dict(device=device, dtype=torch.float64)
    bjerrum, kap2 = _constants(ionic)
    kap = math.sqrt(kap2)
    nx, ny, nz = dims
    co = [torch.arange(n, **f64) * h + (-(n - 1) * h / 2.0) for n in dims]
    host = [c.cpu().numpy() for c in co]
    inside = torch.zeros((nz, ny, nx), device=device, dtype=torch.bool)
    excl = torch.zeros_like(inside)
    src = np.zeros((nz, ny, nx))
    for ax, ay, az, r, q in atoms:
        re = r + 2.0
        cut, cell = [], []
        for c, a in zip(host, (ax, ay, az)):
            cut.append(slice(max(0, int(np.searchsorted(c, a - re)) - 1),
                             int(np.searchsorted(c, a + re)) + 1))
            g = (a - c[0]) / h
            cell.append((int(math.floor(g)), g - math.floor(g)))
        dx, dy, dz = (c[s] - a for c, s, a in zip(co, cut, (ax, ay, az)))
        d2 = ((dx * dx)[None, None, :] + (dy * dy)[None, :, None]) + (dz * dz)[:, None, None]
        box = cut[2], cut[1], cut[0]
        inside[box] |= d2 <= r * r
        excl[box] |= d2 <= re * re
        if all(0 <= c <= n - 2 for (c, _), n in zip(cell, dims)):
            (i, u), (j, v), (k, w) = cell
            wt = np.multiply.outer(np.multiply.outer([1 - w, w], [1 - v, v]), [1 - u, u])
            src[k:k + 2, j:j + 2, i:i + 2] += 4.0 * math.pi * bjerrum * q * wt / h ** 3
    eps = _pick(inside, 2.0, 78.54)
    face = []
    for d in (2, 1, 0):
        up = torch.cat([eps.narrow(d, 1, eps.shape[d] - 1),
                        eps.narrow(d, eps.shape[d] - 1, 1)], d)
        face.append(2 * eps * up / (eps + up))
    u = torch.zeros((nz, ny, nx), **f64)
    at = torch.as_tensor(atoms, **f64)
    amp = bjerrum * at[:, 4] / (78.54 * (1.0 + kap * at[:, 3])) * torch.exp(kap * at[:, 3])
    for d in range(3):
        for side in (0, -1):
            ax = [co[2], co[1], co[0]]
            ax[d] = ax[d][side:][:1] if side else ax[d][:1]
            tot = torch.zeros([len(c) for c in ax], **f64)
            for s in range(0, len(at), 64):
                p, m = at[s:s + 64], amp[s:s + 64]
                r2 = sum((ax[e].view([-1 if e == f else 1 for f in range(3)] + [1])
                          - p[:, 2 - e]) ** 2 for e in range(3))
                r = torch.sqrt(r2)
                tot += (m * torch.exp(-kap * r) / r).sum(-1)
            u.select(d, side if side else 0).copy_(tot.select(d, 0))
    return dict(x=co[0], y=co[1], z=co[2], a=face, cc=_pick(excl, 0.0, 78.54 * kap2),
                f=torch.as_tensor(src, **f64), u=u, h=h)


def _driver_arrays(inp):
    """The driver's argument list: coordinates, the two planes of each pair
    of faces at the front of its (n, n, 4) array, a1cf-a3cf, ccf, fcf, tcf."""
    def flat(t):
        return np.ascontiguousarray(t.cpu().numpy()).reshape(-1)

    u = inp["u"]
    faces = []
    for d in (2, 1, 0):
        g = torch.cat([u.select(d, 0).reshape(-1), u.select(d, -1).reshape(-1)])
        faces.append(np.concatenate([flat(g), np.zeros(g.numel())]))
    return ([flat(inp[k]) for k in "xyz"] + faces + [flat(a) for a in inp["a"]]
            + [flat(inp["cc"]), flat(inp["f"]), np.zeros(u.numel())])


def _apply(inp, v):
    """The flux-balance operator (without the ion term) at interior nodes,
    zero on the boundary."""
    out = torch.zeros_like(v)
    for d, a in zip((2, 1, 0), inp["a"]):
        n = v.shape[d]
        flux = inp["h"] * a.narrow(d, 0, n - 1) * (v.narrow(d, 1, n - 1) - v.narrow(d, 0, n - 1))
        out.narrow(d, 0, n - 1).sub_(flux)
        out.narrow(d, 1, n - 1).add_(flux)
    return _zero_faces(out)


def _zero_faces(v):
    for d in range(3):
        v.select(d, 0).zero_()
        v.select(d, -1).zero_()
    return v


def _cg(inp, ion, rhs, tol, most=8000):
    """Solves (A + ion) v = rhs on the interior, v = 0 on the boundary."""
    diag = ion.clone()
    for d, a in zip((2, 1, 0), inp["a"]):
        diag += inp["h"] * a
        diag.narrow(d, 1, a.shape[d] - 1).add_(inp["h"] * a.narrow(d, 0, a.shape[d] - 1))
    v, r = torch.zeros_like(rhs), rhs.clone()
    z = r / diag
    p, rz = z.clone(), (r * z).sum()
    goal = float(r.norm()) * tol
    for it in range(most):
        q = _apply(inp, p) + ion * p
        _zero_faces(q)
        al = rz / (p * q).sum()
        v += al * p
        r -= al * q
        if it % 40 == 39 and not float(r.norm()) > goal:
            break
        z = r / diag
        new = (r * z).sum()
        p.mul_(new / rz).add_(z)
        rz = new
    return v


def _potential(dims, h, ionic, atoms, nonlinear, device):
    inp = _assemble(dims, h, ionic, atoms, device)
    h3 = h ** 3
    cc = h3 * inp["cc"]
    u = inp["u"].clone()
    u += _cg(inp, cc, _zero_faces(h3 * inp["f"] - _apply(inp, u) - cc * u), 1e-13)
    if nonlinear:
        for _ in range(40):
            w = u.clamp(-85.0, 85.0)
            r = _zero_faces(h3 * inp["f"] - _apply(inp, u) - cc * torch.sinh(w))
            step = _cg(inp, cc * torch.cosh(w), r, 1e-6)
            u += step
            if float(step.abs().max()) <= 1e-12 * float(u.abs().max()):
                break
    return u.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "residual":
        ac, cc, fc, x = _residual_inputs(case, seed, device)
        r = fc - (ac[0] + cc) * x
        for p, d in ((1, 2), (2, 1), (3, 0)):
            r += ac[p] * torch.roll(x, -1, d) + torch.roll(ac[p], 1, d) * torch.roll(x, 1, d)
        _zero_faces(r)
        return {"r": r, "l1": r.abs().sum().reshape(1)}
    if kind == "serve":
        return {"u": [_potential((n, n, n), case["h"], case["ionic"], atoms, False, device)
                      for n, _, atoms in _requests(case, seed)], "iters": None}
    atoms = _molecule(case["natoms"], case["radius"], case["charges"], seed)
    if kind == "dropin":
        dims = case["nx"], case["ny"], case["nz"]
        return {"u": _potential(dims, case["h"], case["ionic"], atoms, False, device),
                "rwork": None, "iters": None}
    n = case["n"]
    return {"u": _potential((n, n, n), case["h"], case["ionic"], atoms, kind == "newton", device),
            "iters": None}
