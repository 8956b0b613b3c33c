"""Timed cases: the calls a T-FlowS host makes of this library, with their inputs.

A T-FlowS outer iteration assembles and solves, in turn, the mixture fraction
(CalcZmix, CG), the three velocity components (NewUVW, BiCG) and the pressure
correction (CalcPS, CG with a cap of 800), then corrects the velocities and the
face fluxes (CorUVW).  The cases are those assemblies and those solves, over the
sizes of this repository's tests and benchmarks: from the few thousand cells of
a test mesh to 256^3.

Solves that end at their cap return x, the residual vector and the two norms;
solves that end at their tolerance return x alone, because the iteration they end
at may shift by one with the rounding of the dot products.
"""
import functools
import math
import random

import numpy as np
import torch

import __graft_entry__

F64 = torch.float64
TINY = 1.0e-64
CFL = 20.0


def _pkg():
    return __graft_entry__.load()


def _dev():
    return torch.device("cuda")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a test mesh (cavity, two materials, 12^3 boxes): the whole solve is launch latency
        {"name": "cg_tiny", "kind": "cg", "nx": 17, "ny": 12, "nz": 11, "mesh": "channel", "prec": 1, "cap": 2000,
         "rtol": 1e-8},
        # the Fortran host's own call, host arrays in and out, at the 32^3 size of the parity runs
        {"name": "dropin_32", "kind": "dropin", "nx": 32, "ny": 32, "nz": 32, "mesh": "channel", "prec": 1,
         "method": "cg", "cap": 2000, "rtol": 1e-8},
        # an ordinary mesh whose lines are no multiple of anything
        {"name": "cg_ragged", "kind": "cg", "nx": 83, "ny": 61, "nz": 97, "mesh": "channel", "prec": 1, "cap": 250,
         "rtol": 0.0},
        # the pressure correction of the 128^3 channel (the benchmark's system), FP64
        {"name": "cg_128", "kind": "cg", "nx": 128, "ny": 128, "nz": 128, "mesh": "channel", "prec": 1, "cap": 400,
         "rtol": 0.0},
        # the same with FP32 iterations and FP64 residual replacement (the benchmark's headline solver)
        {"name": "mixed_128", "kind": "mixed", "nx": 128, "ny": 128, "nz": 128, "mesh": "channel", "prec": 1,
         "cap": 450, "interval": 75},
        # the largest mesh, wall-clustered 256^3: streamed from HBM
        {"name": "cg_wall_256", "kind": "cg", "nx": 256, "ny": 256, "nz": 256, "mesh": "wall", "prec": 1, "cap": 60,
         "rtol": 0.0},
        # DIC preconditioning on a wall-clustered mesh
        {"name": "dic_wall", "kind": "cg", "nx": 128, "ny": 112, "nz": 96, "mesh": "wall", "prec": 2, "cap": 40,
         "rtol": 0.0},
        # CGS on a nonsymmetric momentum matrix of a randomly numbered mesh
        {"name": "cgs_renumbered", "kind": "cgs", "nx": 80, "ny": 72, "nz": 88, "prec": 1, "cap": 2000,
         "rtol": 1e-9, "mixed": False},
        # many uneven pressure systems at once
        {"name": "batch", "kind": "batch", "count": 32, "nmin": 2000, "nmax": 200000, "cap": 60, "shape_seed": 3},
        # a differentiable solve: forward, adjoint and the gradients of the values and of b
        {"name": "adjoint", "kind": "adjoint", "nx": 48, "ny": 40, "nz": 44, "mesh": "channel", "cap": 20000,
         "rtol": 1e-11},
        # the momentum and mixture-fraction assemblies of one outer iteration
        {"name": "transport_assembly", "kind": "transport", "nx": 128, "ny": 112, "nz": 96, "scheme": "SMART",
         "inert": "LIN"},
        # the pressure assembly before the solve, the correction and the CFL monitor after it, on a ragged mesh
        {"name": "pressure_assembly", "kind": "pressure", "nx": 131, "ny": 89, "nz": 107},
    ]


def _box(rng, lo, hi):
    """Three edge lengths of a box of about exp(U(log lo, log hi)) cells."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    a = [rng.uniform(1.0, 2.5) for _ in range(3)]
    s = (n / (a[0] * a[1] * a[2])) ** (1.0 / 3.0)
    e = [max(6, int(round(v * s))) for v in a]
    if rng.random() < 0.35:                        # lines of whole wavefronts, as the tuned meshes have
        e[0] = max(64, (e[0] + 32) // 64 * 64)
        e[1] = max(6, e[1] // 2 * 2)
        e[2] = max(6, e[2] // 2 * 2)
    while e[0] * e[1] * e[2] > 1.3 * hi:
        k = e.index(max(e[1:])) if max(e[1:]) > 6 else 0
        e[k] = max(6, int(e[k] * 0.8))
    return dict(nx=e[0], ny=e[1], nz=e[2])


def draw(rng):
    kind = rng.choice(["cg", "cg", "cg", "mixed", "mixed", "dic", "dropin", "cgs", "batch", "adjoint", "transport",
                       "transport", "pressure", "pressure"])
    mesh = rng.choice(["channel", "wall"])
    if kind == "cg":
        c = _box(rng, 1.5e3, 8e6)
        n, edge = c["nx"] * c["ny"] * c["nz"], max(c["nx"], c["ny"], c["nz"])
        if n < 3e4:                                # small systems are solved to their tolerance
            return dict(c, kind="cg", mesh="channel", prec=1, rtol=1e-8, cap=4000)
        return dict(c, kind="cg", mesh=mesh, prec=1, rtol=0.0,
                    cap=rng.randint(20, max(25, min(300, 2 * edge, int(6e8 / n)))))
    if kind == "mixed":
        c = _box(rng, 2e5, 6e6)
        n = c["nx"] * c["ny"] * c["nz"]
        return dict(c, kind="mixed", mesh="channel", prec=1, cap=rng.randint(100, max(120, min(450, int(6e8 / n)))),
                    interval=rng.choice([50, 75, 100]))
    if kind == "dic":
        return dict(_box(rng, 2e4, 1.4e6), kind="cg", mesh=mesh, prec=2, cap=rng.randint(15, 40), rtol=0.0)
    if kind == "dropin":
        return dict(_box(rng, 2e3, 2e5), kind="dropin", mesh="channel", prec=1, method=rng.choice(["cg", "bicg"]),
                    cap=4000, rtol=1e-8)
    if kind == "cgs":
        return dict(_box(rng, 3e4, 6e5), kind="cgs", prec=1, cap=2000, rtol=1e-9, mixed=rng.random() < 0.4)
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(6, 40), nmin=rng.randint(2000, 6000),
                    nmax=rng.randint(30000, 200000), cap=rng.randint(25, 60), shape_seed=rng.randint(10, 10 ** 6))
    if kind == "adjoint":
        return dict(_box(rng, 1e4, 1.5e5), kind="adjoint", mesh="channel", cap=20000, rtol=1e-11)
    if kind == "transport":
        return dict(_box(rng, 2e4, 1.8e6), kind="transport", scheme=rng.choice(["YES", "SMART", "MINMOD"]),
                    inert=rng.choice(["LIN", "PAR"]))
    return dict(_box(rng, 2e4, 2.2e6), kind="pressure")


# ---------------------------------------------------------------------------
# matrices of box meshes, on the GPU: neighbours in the order -z -y -x self +x
# +y +z, as (n, 7) columns (-1: none) and values
# ---------------------------------------------------------------------------
def _shape(c):
    return c["nx"], c["ny"], c["nz"]


def _neighbours(shape):
    nx, ny, nz = shape
    n = nx * ny * nz
    c = torch.arange(n, dtype=torch.int64, device=_dev())
    i, j, k = c % nx, (c // nx) % ny, c // (nx * ny)
    cols = torch.stack([c - nx * ny, c - nx, c - 1, c, c + 1, c + nx, c + nx * ny], dim=1)
    ok = torch.stack([k > 0, j > 0, i > 0, torch.ones_like(i, dtype=torch.bool), i < nx - 1, j < ny - 1, k < nz - 1],
                     dim=1)
    return torch.where(ok, cols, torch.full_like(cols, -1))


def _smooth(shape, gen, lo, hi):
    """A smooth positive cell field between about lo and hi."""
    nx, ny, nz = shape
    f = torch.zeros((nz, ny, nx), dtype=F64, device=_dev())
    for _ in range(3):
        k = [0.5 + 2.5 * float(torch.rand((), generator=gen)) for _ in range(3)]
        ph = [2 * math.pi * float(torch.rand((), generator=gen)) for _ in range(3)]
        a = [torch.sin(math.pi * k[d] * torch.linspace(0, 1, m, dtype=F64, device=_dev()) + ph[d])
             for d, m in enumerate((nx, ny, nz))]
        f += a[2][:, None, None] * a[1][None, :, None] * a[0][None, None, :] / 3.0
    return (0.5 * (lo + hi) + 0.5 * (hi - lo) * f).reshape(-1)


def _gens(seed):
    cpu = torch.Generator().manual_seed(int(seed))
    dev = torch.Generator(device=_dev()).manual_seed(int(seed) + 77)
    return cpu, dev


def _pressure(shape, mesh, seed):
    """CalcPS.f90:77-94: a_f = |S|/d times the mean of the two cells' V/Asave; cell 1 pinned."""
    mg = _pkg().meshgen
    box = mg.wall_pressure_mesh(shape) if mesh == "wall" else mg.channel_mesh(*shape)
    nx, ny, nz = shape
    cpu, _ = _gens(seed)
    va = _smooth(shape, cpu, 0.6, 1.6).reshape(nz, ny, nx)
    d = [torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device=_dev()) for a in box.spacings()]
    x = [torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device=_dev()) for a in box.centres()]
    area = [d[2][:, None, None] * d[1][None, :, None], d[2][:, None, None] * d[0][None, None, :],
            d[1][None, :, None] * d[0][None, None, :]]
    vals = torch.zeros((nz, ny, nx, 7), dtype=F64, device=_dev())
    for dim, (axis, lo, hi) in enumerate(((2, 2, 4), (1, 1, 5), (0, 0, 6))):
        m = shape[dim]
        v = 0.5 * (va.narrow(axis, 0, m - 1) + va.narrow(axis, 1, m - 1))
        gap = torch.diff(x[dim]).reshape([-1 if a == axis else 1 for a in range(3)])
        ar = area[dim].expand(nz, ny, nx).narrow(axis, 0, m - 1)
        a = ar / gap * v
        vals[..., hi].narrow(axis, 0, m - 1).copy_(-a)
        vals[..., lo].narrow(axis, 1, m - 1).copy_(-a)
    vals[..., 3] = -(vals[..., :3].sum(-1) + vals[..., 4:].sum(-1))
    vals[0, 0, 0, 3] += float(area[0][0, 0, 0] / (0.5 * d[0][0]))
    return _neighbours(shape), vals.reshape(-1, 7)


def _transport(shape, seed):
    """NewUVW.f90:356-367, 447-449 on a unit cube: upwind convection by a velocity whose components do not
    vary along themselves, diffusion 1e-3, the time term of CFL 20."""
    nx, ny, nz = shape
    cpu, _ = _gens(seed)
    h = [1.0 / m for m in shape]
    g = [torch.linspace(0.5 * s, 1 - 0.5 * s, m, dtype=F64, device=_dev()) for s, m in zip(h, shape)]
    ph = [2 * math.pi * float(torch.rand((), generator=cpu)) for _ in range(6)]
    X, Y, Z = g[0][None, None, :], g[1][None, :, None], g[2][:, None, None]
    tau = 2 * math.pi
    vel = [0.5 * torch.sin(tau * Y + ph[0]) + 0.5 * torch.cos(tau * Z + ph[1]),
           0.5 * torch.sin(tau * Z + ph[2]) + 0.5 * torch.cos(tau * X + ph[3]),
           0.5 * torch.sin(tau * X + ph[4]) + 0.5 * torch.cos(tau * Y + ph[5])]
    area = [h[1] * h[2], h[0] * h[2], h[0] * h[1]]
    vals = torch.zeros((nz, ny, nx, 7), dtype=F64, device=_dev())
    for dim, (axis, lo, hi) in enumerate(((2, 2, 4), (1, 1, 5), (0, 0, 6))):
        m = shape[dim]
        F = (vel[dim].expand(nz, ny, nx) * area[dim]).narrow(axis, 0, m - 1)
        D = 1e-3 * area[dim] / h[dim]
        a12, a21 = -torch.clamp(F, max=0.0), torch.clamp(F, min=0.0)
        vals[..., hi].narrow(axis, 0, m - 1).copy_(-(a12 + D))
        vals[..., lo].narrow(axis, 1, m - 1).copy_(-(a21 + D))
        vals[..., 3].narrow(axis, 0, m - 1).add_(a21 + D)
        vals[..., 3].narrow(axis, 1, m - 1).add_(a12 + D)
    vals[..., 3] += h[0] * h[1] * h[2] / (CFL * min(h))
    return _neighbours(shape), vals.reshape(-1, 7)


def _renumber(cols, vals, seed):
    """Cell c becomes row perm[c]; each row's columns ascend, as TopolM sorts them."""
    n = cols.shape[0]
    perm = torch.from_numpy(np.random.default_rng(int(seed)).permutation(n)).to(_dev())
    new = torch.where(cols < 0, torch.full_like(cols, n), perm[cols.clamp(min=0)])
    new, order = torch.sort(new, dim=1)
    vals = torch.gather(vals, 1, order)
    inv = torch.empty_like(perm)
    inv[perm] = torch.arange(n, device=_dev())
    new = torch.where(new == n, torch.full_like(new, -1), new)
    return new[inv], vals[inv]


def _csr(cols, vals):
    """The T-FlowS arrays (1-based, NONZ = nnz + 1) on the GPU."""
    n = cols.shape[0]
    ok = cols >= 0
    counts = ok.sum(1)
    acol = torch.ones(n + 1, dtype=torch.int32, device=_dev())
    acol[1:] = (torch.cumsum(counts, 0) + 1).to(torch.int32)
    nnz = int(counts.sum())
    arow = torch.zeros(nnz + 1, dtype=torch.int32, device=_dev())
    arow[:nnz] = (cols[ok] + 1).to(torch.int32)
    aval = torch.zeros(nnz + 1, dtype=F64, device=_dev())
    aval[:nnz] = vals[ok]
    rows = torch.arange(n, device=_dev())
    before = (ok & (cols < rows[:, None])).sum(1)
    adia = (acol[:-1].to(torch.int64) + before).to(torch.int32)
    return n, nnz + 1, acol, arow, adia, aval


def _rhs(n, seed, mean_free=True):
    _, dev = _gens(seed)
    b = torch.rand(n, dtype=F64, device=_dev(), generator=dev) * 2.0 - 1.0
    return b - b.mean() if mean_free else b


def _batch_shapes(c):
    r = random.Random(c["shape_seed"])
    out = []
    for _ in range(c["count"]):
        n = math.exp(r.uniform(math.log(c["nmin"]), math.log(c["nmax"])))
        a = [r.uniform(1.0, 4.0) for _ in range(3)]
        s = (n / (a[0] * a[1] * a[2])) ** (1.0 / 3.0)
        out.append(tuple(max(3, int(round(v * s))) for v in a))
    return out


def _matrix(c, seed):
    if c["kind"] == "cgs":
        return _renumber(*_transport(_shape(c), seed), seed=c["nx"] + 1000 * c["ny"])
    cols, vals = _pressure(_shape(c), c["mesh"], seed)
    if c["kind"] == "adjoint":                     # a mesh in no particular order
        return _renumber(cols, vals, seed=c["nx"] + 1000 * c["ny"])
    return cols, vals


# ---------------------------------------------------------------------------
# box meshes for the assemblies: faces x, y, z, then the six sides of a channel
# (inflow, outflow, two walls, two symmetry planes)
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=2)
def _mesh(shape):
    """Faces, geometry, pattern and boundary types, as the mesh files would give them."""
    mg = _pkg().meshgen
    box = mg.channel_mesh(shape[0], shape[1], shape[2], 1.05)
    nx, ny, nz = shape
    n = nx * ny * nz
    dev = _dev()
    gen = torch.Generator(device=dev).manual_seed(11)
    cols = _neighbours(shape)
    ok = cols >= 0
    counts = ok.sum(1)
    start = torch.cumsum(counts, 0) - counts
    pos = start[:, None] + torch.cumsum(ok.to(torch.int64), 1) - 1            # 0-based entry of each slot
    d = [torch.as_tensor(np.ascontiguousarray(a), dtype=F64, device=dev) for a in box.spacings()]
    d3 = [d[0][None, None, :].expand(nz, ny, nx).reshape(-1), d[1][None, :, None].expand(nz, ny, nx).reshape(-1),
          d[2][:, None, None].expand(nz, ny, nx).reshape(-1)]
    cid = torch.arange(n, device=dev).reshape(nz, ny, nx)
    c1, c2, s1, s2, axis_of, sign, gap, bc = [], [], [], [], [], [], [], []
    for dim, (axis, lo, hi) in enumerate(((2, 2, 4), (1, 1, 5), (0, 0, 6))):
        a = cid.narrow(axis, 0, shape[dim] - 1).reshape(-1)
        b = cid.narrow(axis, 1, shape[dim] - 1).reshape(-1)
        c1.append(a); c2.append(b); s1.append(pos[a, hi]); s2.append(pos[b, lo])
        axis_of.append(torch.full_like(a, dim)); sign.append(torch.ones_like(a)); bc.append(torch.zeros_like(a))
        gap.append(0.5 * (d3[dim][a] + d3[dim][b]))
    sides = (("inflow", 0, 0, -1), ("outflow", 0, -1, 1), ("wall", 1, 0, -1), ("wall", 1, -1, 1),
             ("symmetry", 2, 0, -1), ("symmetry", 2, -1, 1))
    nbc = 0
    for name, dim, at, sg in sides:
        a = cid.select(2 - dim, at if at == 0 else shape[dim] - 1).reshape(-1)
        c1.append(a); c2.append(-(nbc + 1 + torch.arange(a.numel(), device=dev)) - 1)
        nbc += a.numel()
        s1.append(torch.full_like(a, -1)); s2.append(torch.full_like(a, -1))
        axis_of.append(torch.full_like(a, dim)); sign.append(torch.full_like(a, sg))
        bc.append(torch.full_like(a, mg.BC_CODES[name])); gap.append(0.5 * d3[dim][a])
    c1, c2, s1, s2 = (torch.cat(v) for v in (c1, c2, s1, s2))
    axis_of, sign, gap, bc = (torch.cat(v) for v in (axis_of, sign, gap, bc))
    ns = c1.numel()
    inner = c2 >= 0
    c1f, c2f = c1 + 1, torch.where(inner, c2 + 1, c2 + 1)                      # boundary cells -1 .. -NbC
    tilt = 0.1 * (2 * torch.rand((2, 3, ns), dtype=F64, device=dev, generator=gen) - 1)
    unit = torch.nn.functional.one_hot(axis_of, 3).T.to(F64)
    ar = torch.stack([d3[1] * d3[2], d3[0] * d3[2], d3[0] * d3[1]])[axis_of, c1]
    S = (unit + tilt[0] * (1 - unit)) * ar * sign
    D = (unit + tilt[1] * (1 - unit)) * gap * sign
    f = torch.where(inner, 0.5 + 0.1 * tilt[0].sum(0), torch.ones(ns, dtype=F64, device=dev))
    volume = torch.zeros(nbc + n + 1, dtype=F64, device=dev)
    volume[nbc + 1:] = d3[0] * d3[1] * d3[2]
    typebc = torch.zeros(nbc + n + 1, dtype=torch.int32, device=dev)
    typebc[nbc + c2f[~inner]] = bc[~inner].to(torch.int32)
    sidec = torch.zeros((3, ns), dtype=torch.int32, device=dev)
    sidec[1], sidec[2] = c1f.to(torch.int32), c2f.to(torch.int32)
    sidaij = torch.stack([s1 + 1, s2 + 1]).to(torch.int32)
    nnz = int(counts.sum())
    host = lambda t: np.ascontiguousarray(t.cpu().numpy())                      # noqa: E731
    acol = torch.cat([start, start.new_full((1,), nnz)]) + 1
    arow = torch.zeros(nnz + 1, dtype=torch.int32, device=dev)
    arow[:nnz] = (cols[ok] + 1).to(torch.int32)
    adia = pos[:, 3] + 1
    empty = np.zeros(0)
    case = mg.CalcPSCase(shape, n, nbc, ns, nnz + 1, 1, 1e-2, host(sidec), host(sidaij), host(acol.to(torch.int32)),
                         host(arow), host(adia.to(torch.int32)), host(typebc), *(host(t) for t in S),
                         *(host(t) for t in D), host(f), host(volume), *([empty] * 11))
    keep = {"c1": c1f + nbc, "c2": c2f + nbc, "inner": inner, "bc": bc, "s1": s1, "s2": s2, "S": S, "D": D, "f": f,
            "volume": volume, "adia": pos[:, 3], "nnz": nnz, "n": n, "nbc": nbc, "ns": ns}
    keep["scoef"] = (S * S).sum(0) / (S * D).sum(0)
    return case, keep


def _cell_fields(g, seed, names):
    """Smooth cell arrays (-NbC:NC) with a little noise; cell 0 is no cell."""
    _, dev = _gens(seed)
    m = g["nbc"] + g["n"] + 1
    t = torch.arange(m, dtype=F64, device=_dev())
    out = {}
    for name, mean, amp in names:
        ph = torch.rand(3, dtype=F64, device=_dev(), generator=dev)
        a = torch.sin(t * (0.011 + 0.01 * ph[0]) + 6 * ph[1]) * torch.cos(t * 1e-4 * (1 + ph[2]))
        a = mean + amp * (a + 0.2 * (2 * torch.rand(m, dtype=F64, device=_dev(), generator=dev) - 1))
        a[g["nbc"]] = 0.0
        out[name] = a
    return out


def _pressure_fields(g, seed):
    dt = 1e-2
    v = _cell_fields(g, seed, [("rho_n", 1.0, 0.05), ("rho_o", 1.0, 0.05), ("rho_oo", 1.0, 0.05), ("u", 1.0, 0.3),
                               ("v", 0.0, 0.2), ("w", 0.0, 0.2), ("p", 0.0, 0.5), ("px", 0.0, 0.4), ("py", 0.0, 0.4),
                               ("pz", 0.0, 0.4), ("wa", 1.6, 0.1), ("pp", 0.0, 0.02)])
    v["asave"] = g["volume"] / dt * v.pop("wa")
    return v


SCHEMES = {"YES": 10, "SMART": 24, "MINMOD": 23}
INERT = {"LIN": 4, "PAR": 5}
UVW = {1: (("ux", "uy", "uz", "vx", "wx", "vy", "wz"), (0, 1, 2), "px"),
       2: (("vy", "vx", "vz", "uy", "wy", "ux", "wz"), (1, 0, 2), "py"),
       3: (("wz", "wx", "wy", "uz", "vz", "ux", "vy"), (2, 0, 1), "pz")}


def _transport_fields(g, seed):
    names = [("rho_n", 1.0, 0.05), ("rho_o", 1.0, 0.05), ("rho_oo", 1.0, 0.05), ("px", 0.0, 0.4), ("py", 0.0, 0.4),
             ("pz", 0.0, 0.4), ("z", 0.5, 0.3), ("z_o", 0.5, 0.3), ("z_oo", 0.5, 0.3), ("src_z", 0.0, 0.05)]
    names += [(a + b, 0.1, 0.4) for a in "uvwz" for b in "xyz"]
    for k, mean in (("u", 1.0), ("v", 0.0), ("w", 0.0)):
        names += [(k, mean, 0.3), (k + "_o", mean, 0.3), (k + "_oo", mean, 0.3), ("src_" + k, 0.0, 0.1)]
    v = _cell_fields(g, seed, names)
    f = g["f"]
    flux = sum((f * v[k][g["c1"]] + (1 - f) * v[k][g["c2"]]) * g["S"][q] for q, k in enumerate("uvw"))
    flux[(g["bc"] == 2) | (g["bc"] == 4)] = 0.0    # no flux through walls and symmetry planes
    v["flux_u"] = flux
    return v


def _transport_params(c):
    mg = _pkg().meshgen
    inert = INERT[c["inert"]]
    uvw = [mg.uvw_params(var=q, blend=[10], blend_tem=[10], urf=0.7, inert=inert) for q in (1, 2, 3)]
    zmix = mg.uvw_params(blend_tem=[SCHEMES[c["scheme"]]], urf=0.8, visc=2e-3, inert=inert)
    return uvw, zmix


# ---------------------------------------------------------------------------
# prepare, run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kr = _pkg().krylov
    k = case["kind"]
    st = {"case": case}
    if k in ("cg", "mixed", "cgs", "adjoint"):
        cols, vals = _matrix(case, seed)
        n, nonz, acol, arow, adia, aval = _csr(cols, vals)
        del cols, vals
        st["system"] = kr.DeviceSystem.from_device(n, nonz, acol, arow, adia, aval)
        st["b"] = _rhs(n, seed, k != "cgs")
        st["x"], st["r"] = torch.zeros_like(st["b"]), torch.empty_like(st["b"])
        st["tol"] = case.get("rtol", 0.0) * float(torch.linalg.vector_norm(st["b"]))
        if k == "adjoint":
            st["aval"] = aval
            st["gx"] = _rhs(n, seed + 5000)
    elif k == "dropin":
        n, nonz, acol, arow, adia, aval = _csr(*_matrix(case, seed))
        st["args"] = (n, 0, nonz, *(t.cpu().numpy() for t in (aval, acol, arow, adia)), np.zeros(1))
        st["b"] = _rhs(n, seed).cpu().numpy()
        st["tol"] = case["rtol"] * float(np.linalg.norm(st["b"]))
        st["x"], st["r"] = np.zeros(n + 1), np.empty(n)
    elif k == "batch":
        mats, rhs = [], []
        T = _pkg().meshgen.TFlowSMatrix
        for q, shape in enumerate(_batch_shapes(case)):
            n, nonz, *a = _csr(*_pressure(shape, "channel", seed * 100 + q))
            mats.append(T(n, nonz, *(t.cpu().numpy() for t in a)))
            rhs.append(_rhs(n, seed * 100 + q))
        st["batch"] = kr.DeviceBatch(mats)
        st["b"] = torch.cat(rhs)
        st["x"], st["r"] = torch.zeros_like(st["b"]), torch.empty_like(st["b"])
    else:
        mesh, g = _mesh(_shape(case))
        dc = st["handle"] = kr.DeviceCalcPS(mesh)
        dc.uvw_setup({"scoef": g["scoef"].cpu().numpy(), "ff": g["f"].cpu().numpy(),
                      "material": np.ones(g["nbc"] + g["n"] + 1, np.int32), "nmaterials": 1})
        new = lambda m: torch.zeros(m, dtype=F64, device=_dev())               # noqa: E731
        ncell = g["nbc"] + g["n"] + 1
        if k == "pressure":
            st["fields"] = _pressure_fields(g, seed)
            st["out"] = {"aval": new(g["nnz"] + 1), "b": new(g["n"]), "flux": new(g["ns"]), "abou": new(g["nbc"])}
            st["vel"] = [new(ncell) for _ in range(3)]
            st["b2"] = new(g["n"])
        else:
            v = _transport_fields(g, seed)
            st["params"], st["zparams"] = _transport_params(case)
            st["inputs"] = [[v["rho_n"], v["rho_o"], v["rho_oo"], v[a], v[a + "_o"], v[a + "_oo"], v["src_" + a],
                             v[UVW[q + 1][2]], *(v[s] for s in UVW[q + 1][0]), v["flux_u"], None]
                            for q, a in enumerate("uvw")]
            st["zinputs"] = [v["rho_n"], v["rho_o"], v["rho_oo"], v["z"], v["z_o"], v["z_oo"], v["src_z"], v["zx"],
                             v["zy"], v["zz"], v["flux_u"], None]
            st["outs"] = [{"aval": new(g["nnz"] + 1), "b": new(g["n"]), "abou": new(g["nbc"]), "asave": new(ncell),
                           "rhoui": new(ncell)} for _ in range(3)]
            st["zout"] = {"aval": new(g["nnz"] + 1), "b": new(g["n"]), "abou": new(g["nbc"]), "rhoz": new(ncell)}
            st["next"] = [new(ncell) for _ in range(4)]
    torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    k = case["kind"]
    kr = _pkg().krylov
    if k == "cg":
        x, r = st["x"].zero_(), st["r"].copy_(st["b"])
        it, ini, fin = st["system"].solve("cg", case["prec"], x, r, case["cap"], st["tol"])
        return {"x": x} if st["tol"] > 0.0 else {"x": x, "r": r, "ini": ini, "fin": fin, "niter": it}
    if k == "mixed":
        x = st["x"].zero_()
        _, ini, _, _ = st["system"].solve_mixed_reliable(case["prec"], x, st["b"], case["cap"], 0.0,
                                                         interval=case["interval"])
        return {"x": x, "ini": ini}
    if k == "cgs":
        x = st["x"].zero_()
        if case["mixed"]:
            st["system"].solve_mixed("cgs", case["prec"], x, st["b"], case["cap"], st["tol"], inner_rtol=1e-3)
        else:
            st["system"].solve("cgs", case["prec"], x, st["r"].copy_(st["b"]), case["cap"], st["tol"])
        return {"x": x}
    if k == "dropin":
        st["x"][:] = 0.0
        st["r"][:] = st["b"]
        getattr(kr, case["method"])(*st["args"], st["x"], st["r"], case["prec"], case["cap"], st["tol"])
        return {"x": st["x"]}
    if k == "batch":
        x, r = st["x"].zero_(), st["r"].copy_(st["b"])
        got = st["batch"].solve("cg", 1, x, r, case["cap"], 0.0)
        return {"x": x, "r": r, "ini": got["ini_res"], "fin": got["fin_res"], "niter": got["niter"]}
    if k == "adjoint":
        from tflows_amd import autograd
        a = st["aval"].detach().requires_grad_(True)
        b = st["b"].detach().requires_grad_(True)
        x = autograd.solve(a, b, st["system"], "cg", 1, case["rtol"], case["cap"])
        ga, gb = torch.autograd.grad(x, (a, b), st["gx"])
        return {"x": x, "grad_a": ga, "grad_b": gb}
    dc = st["handle"]
    if k == "pressure":
        f, vel = st["fields"], st["vel"]
        got = dc.assemble(f, out=st["out"])
        assembled = got["flux"].clone()             # the correction works on Flux in place
        for t, name in zip(vel, "uvw"):
            t.copy_(f[name])
        b2, err2 = dc.correct(f["pp"], got["aval"], got["abou"], *vel, got["flux"], fields=f, b=st["b2"])
        cfl, pe = dc.cfl_peclet(f["rho_n"], got["flux"], 1e-2, 1e-2)
        return {"aval": got["aval"], "b": got["b"], "flux0": assembled, "flux": got["flux"], "errmax": got["errmax"],
                "mean": got["mean"], "vel": vel, "b2": b2, "err2": err2, "cfl": cfl, "pe": pe}
    res = []
    for q in range(3):
        o = dc.assemble_uvw(st["params"][q], st["inputs"][q], out=st["outs"][q])
        dc.uvw_update(o["rhoui"], st["inputs"][q][0], st["next"][q])
        res.append({"aval": o["aval"], "b": o["b"], "rhoui": o["rhoui"], "next": st["next"][q]})
    res[0]["asave"] = st["outs"][0]["asave"]
    o = dc.assemble_zmix(st["zparams"], st["zinputs"], out=st["zout"])
    dc.zmix_update(o["rhoz"], st["zinputs"][0], st["next"][3])
    res.append({"aval": o["aval"], "b": o["b"], "rhoz": o["rhoz"], "next": st["next"][3]})
    return res


# ---------------------------------------------------------------------------
# work and tolerances
# ---------------------------------------------------------------------------
def _faces(shape):
    nx, ny, nz = shape
    return (nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1)


def _sides(shape):
    nx, ny, nz = shape
    return 2 * (ny * nz + nx * nz + nx * ny)


def _iterations(c):
    """Iterations a solve to its tolerance takes, roughly (Jacobi CG on these meshes: a few times the longest line)."""
    if c["kind"] == "cgs":
        return 2.2 * max(_shape(c))
    return 15.0 * max(_shape(c)) * math.sqrt(-math.log10(c["rtol"]) / 8.0)


def work(case):
    """Bytes of one pass: per iteration every distinct matrix value once (a symmetric matrix has one per face and
    one per cell) and x, r, p read and written, q written and read, the preconditioner read; whole arrays once
    for the assemblies."""
    k = case["kind"]
    if k == "batch":
        n = sum(a * b * c for a, b, c in _batch_shapes(case))
        faces = sum(_faces(s) for s in _batch_shapes(case))
        its = case["cap"]
    else:
        n, faces = case["nx"] * case["ny"] * case["nz"], _faces(_shape(case))
        its = case["cap"] if k == "mixed" or (k == "cg" and case["rtol"] == 0.0) else 0
    if k in ("cg", "batch", "mixed", "dropin", "adjoint"):
        w = 4 if k == "mixed" else 8
        if not its:
            its = _iterations(case) * (2 if k == "adjoint" else 1)
        sweeps = 2 if case.get("prec") == 2 else 0
        per = w * (faces + n) + w * 9 * n + sweeps * (w * faces + w * 3 * n)
        return {"bytes": float(its * per), "flops": float(its * (2 * (2 * faces + n) * (1 + sweeps / 2) + 12 * n))}
    if k == "cgs":
        its, w = _iterations(case), 4 if case["mixed"] else 8
        per = 2 * (w * (2 * faces + n) + 4 * 2 * faces) + w * 16 * n
        return {"bytes": float(its * per), "flops": float(its * (4 * (2 * faces + n) + 20 * n))}
    ns, nb = faces + _sides(_shape(case)), _sides(_shape(case))
    cell = 8 * (n + nb)
    if k == "pressure":
        # per face its cells, positions, S, D, f, the flux; per cell the fields; Aval, b
        asm = ns * (16 + 56 + 8) + 12 * cell + 8 * (2 * faces + n) + 8 * n
        cor = ns * (16 + 8 + 8) + 8 * faces + 12 * cell + 4 * cell
        cfl = ns * (8 + 8 * 6) + cell
        return {"bytes": float(asm + cor + cfl), "flops": float(80 * ns + 30 * n)}
    one = ns * (16 + 8 * 10) + 8 * (2 * faces + n) + 2 * 8 * n
    return {"bytes": float(3 * (one + 16 * cell) + one + 11 * cell + 4 * 3 * 8 * n), "flops": float(4 * 120 * ns)}


def tolerance(case):
    """About four times what the largest of a few dozen cases of a kind was off its 64-bit evaluation."""
    k = case["kind"]
    if k == "mixed":                               # FP32 iterations: seen 1e-6 in x
        return {"rel": 5e-6}
    if k in ("transport", "pressure"):             # sums of at most a dozen terms in another order: 2e-16
        return {"rel": 2e-15, "max": 1e-12}
    if k == "adjoint":                             # solved to 1e-11 of b: 1e-11
        return {"rel": 1e-10}
    if k == "cgs" or case.get("rtol", 0.0) > 0.0:  # solved to 1e-8 or 1e-9 of b: 1e-8
        return {"rel": 1e-7}
    return {"rel": 1e-11}                          # a fixed number of FP64 iterations: 6e-13 in r


# ---------------------------------------------------------------------------
# the same results from plain torch in 64 bits
# ---------------------------------------------------------------------------
class _Ell:
    def __init__(self, cols, vals):
        self.idx = cols.clamp(min=0)
        self.vals = torch.where(cols >= 0, vals, torch.zeros_like(vals))
        rows = torch.arange(cols.shape[0], device=cols.device)[:, None]
        self.lower, self.upper = (cols >= 0) & (cols < rows), cols > rows
        self.diag = torch.where(cols == rows, vals, torch.zeros_like(vals)).sum(1)

    def mul(self, p):
        return (self.vals * p[self.idx]).sum(1)


class _Dic:
    """Prec1.f90:51-59 and the sweeps of CG.f90:135-156, level by level (i + j + k of a box)."""

    def __init__(self, A, shape):
        nx, ny, nz = shape
        c = torch.arange(nx * ny * nz, device=A.diag.device)
        lev = c % nx + (c // nx) % ny + c // (nx * ny)
        order = torch.argsort(lev, stable=True)
        self.levels = torch.split(order, torch.bincount(lev).tolist())
        self.lo = [(A.idx[r, :3], torch.where(A.lower[r, :3], A.vals[r, :3], 0.0)) for r in self.levels]
        self.up = [(A.idx[r, 4:], torch.where(A.upper[r, 4:], A.vals[r, 4:], 0.0)) for r in self.levels]
        self.D = torch.zeros_like(A.diag)
        for r, (i, v) in zip(self.levels, self.lo):
            self.D[r] = 1.0 / (A.diag[r] - (self.D[i] * v * v).sum(1))

    def __call__(self, u):
        z = torch.zeros_like(u)
        for r, (i, v) in zip(self.levels, self.lo):
            z[r] = (u[r] - (v * z[i]).sum(1)) * self.D[r]
        z = z / (self.D + TINY)
        for r, (i, v) in zip(reversed(self.levels), reversed(self.up)):
            z[r] = (z[r] - (v * z[i]).sum(1)) * self.D[r]
        return z


def _cg(A, prec, b, cap, tol):
    x, r, p = torch.zeros_like(b), b.clone(), None
    ini = fin = torch.linalg.vector_norm(r)
    rho_old = None
    for it in range(cap):
        z = prec(r)
        rho = torch.dot(r, z)
        p = z.clone() if p is None else z + (rho / rho_old) * p
        q = A.mul(p)
        alfa = rho / torch.dot(p, q)
        x += alfa * p
        r -= alfa * q
        fin = torch.linalg.vector_norm(r)
        if tol > 0.0 and float(fin) < tol:
            break
        rho_old = rho
    return x, r, float(ini), float(fin)


def _cgs(A, b, cap, tol):
    x, r, r2 = torch.zeros_like(b), b.clone(), b.clone()
    q = u2 = rho_old = None
    for _ in range(cap):
        rho = torch.dot(r, r2)
        if q is None:
            u1, u2 = r.clone(), r.clone()
        else:
            beta = rho / rho_old
            u1 = r + beta * q
            u2 = u1 + beta * (q + beta * u2)
        v = A.mul(u2 / A.diag)
        alfa = rho / torch.dot(r2, v)
        q = u1 - alfa * v
        w = (u1 + q) / A.diag
        x += alfa * w
        r -= alfa * A.mul(w)
        if float(torch.linalg.vector_norm(r)) < tol:
            break
        rho_old = rho
    return x


def _exact_pressure(case, seed):
    mesh, g = _mesh(_shape(case))
    v = _pressure_fields(g, seed)
    nb, n, dt = g["nbc"], g["n"], 1e-2
    c1, c2, f, inner, bc = g["c1"], g["c2"], g["f"], g["inner"], g["bc"]
    S, D, V = g["S"], g["D"], g["volume"]
    r1, r2 = f * v["rho_n"][c1], (1 - f) * v["rho_n"][c2]
    mass = sum((r1 * v[k][c1] + r2 * v[k][c2]) * S[q] for q, k in enumerate("uvw"))
    smdpn = (S * S).sum(0) / (S * D).sum(0)
    va = V / torch.where(v["asave"] == 0, torch.ones_like(V), v["asave"])
    a12 = torch.where(inner, 0.5 * smdpn * (va[c1] + va[c2]), smdpn * va[c1])
    dp = sum(0.5 * (v[k][c1] + v[k][c2]) * D[q] for q, k in enumerate(("px", "py", "pz")))
    flux = torch.where(inner, mass + a12 * (v["p"][c1] - v["p"][c2]) + a12 * dp, mass)
    live = inner | (bc == 1) | (bc == 3)
    flux = torch.where(live, flux, torch.zeros_like(flux))
    dg = torch.where(inner | (bc == 3), a12, torch.zeros_like(a12))
    i1, i2 = c1 - nb - 1, c2[inner] - nb - 1
    zero = torch.zeros(n, dtype=F64, device=_dev())
    diag = zero.index_add(0, i1, dg).index_add(0, i2, dg[inner])
    b0 = zero.index_add(0, i1, -flux).index_add(0, i2, flux[inner])
    aval = torch.zeros(g["nnz"] + 1, dtype=F64, device=_dev())
    aval[g["s1"][inner]] = -a12[inner]
    aval[g["s2"][inner]] = -a12[inner]
    aval[g["adia"]] = diag
    Vc = V[nb + 1:]
    term = Vc / dt * (1.5 * v["rho_n"] - 2.0 * v["rho_o"] + 0.5 * v["rho_oo"])[nb + 1:]
    b = b0 - term
    mean = float((b * Vc).sum() / Vc.sum())
    live_c = slice(nb + 1, None)
    vel = []
    for k, pk in zip("uvw", ("px", "py", "pz")):
        t = v[k].clone()
        t[live_c] -= v[pk][live_c] * Vc / v["asave"][live_c] / v["rho_n"][live_c]
        vel.append(t)
    flux2 = torch.where(inner, flux - (v["pp"][c2] - v["pp"][c1]) * a12, flux)
    b2 = (zero.index_add(0, i1, -flux2).index_add(0, i2, flux2[inner]) - term) / Vc
    rhos = f * v["rho_n"][c1] + (1 - f) * v["rho_n"][c2]
    cfl = (dt * flux2 / (rhos * g["scoef"] * (D * D).sum(0))).abs()[inner].max()
    pe = (flux2 / g["scoef"] / 1e-2).abs()[inner].max()
    return {"aval": aval, "b": b - mean, "flux0": flux, "flux": flux2, "errmax": float(b0.abs().max()), "mean": mean,
            "vel": vel, "b2": b2, "err2": float(b2.abs().max()), "cfl": np.array([float(cfl)]),
            "pe": np.array([float(pe)])}


def _face_value(scheme, g, phi, grad, D, pmin, pmax, flux, phis):
    """Process/ConvScheme.f90:55-118 for the schemes of the cases."""
    if scheme == "YES":
        return phis
    c1, c2, f = g["c1"], g["c2"], g["f"]
    pos = flux > 0.0
    fj = torch.where(pos, 1 - f, f)
    C, Dn = torch.where(pos, c1, c2), torch.where(pos, c2, c1)
    gd = sum(a[C] * D[q] for q, a in enumerate(grad))
    star = torch.where(pos, phi[Dn] - 2 * gd, phi[Dn] + 2 * gd)
    up = torch.maximum(pmin[C], torch.minimum(star, pmax[C]))
    rj = (phi[C] - up) / (phi[Dn] - phi[C] + 1e-16)
    if scheme == "MINMOD":
        lim = fj * torch.clamp(rj, 0.0, 1.0)
    else:
        quick = 0.5 * fj * (1 + fj) + 0.5 * fj * (1 - fj) * rj
        lim = torch.clamp(torch.minimum(torch.minimum(2.0 * rj, quick), torch.ones_like(rj)), min=0.0)
    return phi[C] + lim * torch.where(pos, 1.0, -1.0) * (phi[c2] - phi[c1])


def _exact_equation(g, P, v, names, grads, S, D, pi, scheme, scalar):
    """NewUVW.f90:137-499 and CalcZmix.f90:100-387 for one material."""
    nb, n = g["nbc"], g["n"]
    c1, c2, f, inner, bc = g["c1"], g["c2"], g["f"], g["inner"], g["bc"]
    rho, Fu, V = v["rho_n"], v["flux_u"], g["volume"][nb + 1:]
    phi_n, phi_o, phi_oo, src = (v[k] for k in names)
    phi = rho * phi_n
    i1, i2 = c1 - nb - 1, c2[inner] - nb - 1
    zero = torch.zeros(n, dtype=F64, device=_dev())
    pmax, pmin = phi.clone(), phi.clone()
    for a, b in ((c1[inner], c2[inner]), (c2[inner], c1[inner])):
        pmax.index_reduce_(0, a, phi[b], "amax")
        pmin.index_reduce_(0, a, phi[b], "amin")
    phis = _face_value(scheme, g, phi, grads[:3], D, pmin, pmax, Fu, f * phi[c1] + (1 - f) * phi[c2])
    conv, up = Fu * phis, Fu * torch.where(Fu < 0, phi[c2], phi[c1])
    spread = lambda t: zero.index_add(0, i1, -t).index_add(0, i2, t[inner])     # noqa: E731
    gS = [f * a[c1] + (1 - f) * a[c2] for a in grads]
    if scalar:
        fex = P["visc"] * (gS[0] * S[0] + gS[1] * S[1] + gS[2] * S[2])
    else:
        fex = P["visc"] * (4.0 / 3.0 * gS[0] * S[0] + (gS[1] + gS[3]) * S[1] + (gS[2] + gS[4]) * S[2] -
                           2.0 / 3.0 * (gS[5] + gS[6]) * S[0])
    A0 = P["visc"] * g["scoef"]
    fim = A0 * (gS[0] * D[0] + gS[1] * D[1] + gS[2] * D[2])
    d12, d21 = A0 / rho[c2], A0 / rho[c1]
    a12, a21 = -torch.clamp(Fu, max=0.0), torch.clamp(Fu, min=0.0)
    wall, out = (bc == 1) | (bc == 2), bc == 3
    dg1 = torch.where(inner | wall, a21 + d21, torch.where(out, a21, torch.zeros_like(a21)))
    diag = zero.index_add(0, i1, dg1).index_add(0, i2, (a12 + d12)[inner])
    bb = P["urfc"][0] * (spread(conv) - spread(up))
    bnd = torch.where(wall, (a12 + d12) * phi[c2], torch.where(out, a12 * phi[c2], torch.zeros_like(a12)))
    bb = bb + zero.index_add(0, i1, bnd) - spread(fex - fim)
    cell = slice(nb + 1, None)
    dt = P["dt"]
    if P["inert"] == 4:
        diag = diag + V / dt
        bb = bb + V / dt * v["rho_o"][cell] * phi_o[cell]
    else:
        diag = diag + 1.5 * V / dt
        bb = bb + 2.0 * V / dt * v["rho_o"][cell] * phi_o[cell] - 0.5 * V / dt * v["rho_oo"][cell] * phi_oo[cell]
    bb = bb + src[cell] * V
    if not scalar:
        bb = bb - pi[cell] * V
    bb = bb + diag * (1.0 - P["urf"]) * phi[cell] / P["urf"]
    aval = torch.zeros(g["nnz"] + 1, dtype=F64, device=_dev())
    aval[g["s1"][inner]] = -(a12 + d12)[inner]
    aval[g["s2"][inner]] = -(a21 + d21)[inner]
    aval[g["adia"]] = diag / P["urf"]
    nxt = torch.zeros_like(phi)
    nxt[cell] = phi[cell] / rho[cell]
    if scalar:
        nxt.clamp_(0.0, 1.0)
    asave = torch.zeros_like(phi)
    asave[cell] = diag
    return aval, bb, phi, nxt, asave


def _exact_transport(case, seed):
    _, g = _mesh(_shape(case))
    v = _transport_fields(g, seed)
    uvw, zmix = _transport_params(case)
    res = []
    for q, a in enumerate("uvw"):
        grads, order, pname = UVW[q + 1]
        aval, b, ru, nxt, asave = _exact_equation(g, uvw[q], v, (a, a + "_o", a + "_oo", "src_" + a),
                                                  [v[s] for s in grads], [g["S"][o] for o in order],
                                                  [g["D"][o] for o in order], v[pname], "YES", False)
        res.append({"aval": aval, "b": b, "rhoui": ru, "next": nxt})
        if q == 0:
            res[0]["asave"] = asave
    aval, b, ru, nxt, _ = _exact_equation(g, zmix, v, ("z", "z_o", "z_oo", "src_z"), [v["zx"], v["zy"], v["zz"]],
                                          list(g["S"]), list(g["D"]), None, case["scheme"], True)
    res.append({"aval": aval, "b": b, "rhoz": ru, "next": nxt})
    return res


def exact(case, seed):
    k = case["kind"]
    if k == "pressure":
        return _exact_pressure(case, seed)
    if k == "transport":
        return _exact_transport(case, seed)
    if k == "batch":
        xs, rs, ini, fin = [], [], [], []
        for q, shape in enumerate(_batch_shapes(case)):
            A = _Ell(*_pressure(shape, "channel", seed * 100 + q))
            x, r, i0, f0 = _cg(A, lambda t: t / A.diag, _rhs(A.diag.numel(), seed * 100 + q), case["cap"], 0.0)
            xs.append(x); rs.append(r); ini.append(i0); fin.append(f0)
        return {"x": torch.cat(xs), "r": torch.cat(rs), "ini": np.array(ini), "fin": np.array(fin), "niter": None}
    cols, vals = _matrix(case, seed)
    A = _Ell(cols, vals)
    b = _rhs(A.diag.numel(), seed, k != "cgs")
    prec = _Dic(A, _shape(case)) if case.get("prec") == 2 else (lambda t: t / A.diag) if case.get("prec", 1) == 1 \
        else (lambda t: t.clone())
    if k == "cgs":
        return {"x": _cgs(A, b, case["cap"], 1e-12 * float(torch.linalg.vector_norm(b)))}
    if k == "adjoint":
        x = _cg(A, prec, b, case["cap"], 1e-13 * float(torch.linalg.vector_norm(b)))[0]
        gx = _rhs(A.diag.numel(), seed + 5000)
        lam = _cg(A, prec, gx, case["cap"], 1e-13 * float(torch.linalg.vector_norm(gx)))[0]
        ok = cols >= 0
        rows = torch.arange(cols.shape[0], device=_dev())[:, None].expand_as(cols)
        ga = torch.zeros(int(ok.sum()) + 1, dtype=F64, device=_dev())
        ga[:-1] = -lam[rows[ok]] * x[cols[ok]]
        return {"x": x, "grad_a": ga, "grad_b": lam}
    if k == "mixed":
        x, _, ini, _ = _cg(A, prec, b, case["cap"], 0.0)
        return {"x": x, "ini": ini}
    converged = case["rtol"] > 0.0
    tol = 1e-12 * float(torch.linalg.vector_norm(b)) if converged else 0.0
    x, r, ini, fin = _cg(A, prec, b, 5 * case["cap"] if converged else case["cap"], tol)
    if k == "dropin":
        return {"x": np.concatenate([[0.0], x.cpu().numpy()])}
    return {"x": x} if converged else {"x": x, "r": r, "ini": ini, "fin": fin, "niter": None}
