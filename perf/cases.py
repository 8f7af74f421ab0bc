"""Performance cases of the operator-application library.

A case is one call, or the short chain of calls, that a program using the
library makes over and over: operator applies (FP64 and split-BF16, device and
host cubes), batches of Helmholtz applies, the grid-based FMM potential, the
bubbles' injection, products and potentials of bubble-carrying functions, one
iteration's work of the cube-orbital SCF, and a training pass of the learned
preconditioner.  `listed()` names twelve of them; `draw(rng)` gives others of
the same ranges.

Cubes stay in device memory; outputs are torch views of the library's own
device buffers.  `exact(case, seed)` recomputes a case in 64 bits with torch
alone: the operator matrices by Gauss-Legendre quadrature of the Lagrange
cells, the contractions as dense products, the bubbles point by point.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

import dage_amd
import dage_amd.function3d as f3d
import dage_amd.learned as learned
import dage_amd.scf as scf
from dage_amd._lib import call

PREC = {"fp64": dage_amd.DAGE_PREC_FP64, "bf16x6": dage_amd.DAGE_PREC_BF16X6,
        "bf16x3": dage_amd.DAGE_PREC_BF16X3}


# --------------------------------------------------------------------- cases
def _grid_case(kind, cells, nlip, h, **more):
    return dict(kind=kind, cx=cells[0], cy=cells[1], cz=cells[2], nlip=nlip, h=h, **more)


def _quad(nlin, nlog, tlog):
    return dict(nlin=nlin, nlog=nlog, tlog=float(tlog))


T18, T40, T50 = _quad(10, 8, 1000.0), _quad(20, 20, 500.0), _quad(25, 25, 1000.0)


def listed():
    def c(name, kind, cells, nlip, h, **more):
        return dict(_grid_case(kind, cells, nlip, h, **more), name=name)

    return [
        # the smallest call: one Coulomb apply on a small box (an atom, a test
        # calculation), where the launches count
        c("apply-31", "apply", (5, 5, 5), 7, 0.32, energy=0.0, precision="fp64", **T40),
        # the plain Coulomb apply of an ordinary molecule
        c("apply-97", "apply", (16, 16, 16), 7, 1.0 / 6.0, energy=0.0, precision="fp64", **T40),
        # the Fortran program's call: host cubes in and out, one Helmholtz
        # energy per call, an odd box
        c("host-85x97x73", "host", (14, 16, 12), 7, 1.0 / 6.0, energy=-0.7, precision="fp64",
          **T40),
        # the split-BF16 option on an ordinary cube
        c("bf16x6-129", "apply", (32, 32, 32), 5, 0.15, energy=-0.5, precision="bf16x6", **T40),
        # a density with four atoms' bubbles injected and its potential by the
        # grid-based FMM
        c("gbfmm-241", "gbfmm", (40, 40, 40), 7, 0.1, energy=0.0, boxes=2, lmax=12, atoms=4,
          blmax=4, **T50),
        # one iteration's operators of the SCF on twelve cube orbitals
        c("scf-129", "scf", (32, 32, 32), 5, 0.15, orbitals=12, **T40),
        # orbitals on cubes of uneven sizes, each with its own energy
        c("batch-uneven", "batch", (0, 0, 0), 5, 0.15, sizes="65x4,97x4,129x4,161x4", **T40),
        # a slice of the sweep over the largest cube's orbitals
        c("batch-385", "batch", (0, 0, 0), 7, 0.1, sizes="385x4", **T40),
        # four atoms' bubbles onto a large cube
        c("inject-241", "inject", (40, 40, 40), 7, 0.1, atoms=4, blmax=4),
        # the product of two orbitals that carry bubbles on ten atoms, and its
        # integral (exchange integrals and overlaps are made of these)
        c("product-129", "product", (32, 32, 32), 5, 0.15, atoms=10, blmax=4),
        # the Coulomb potential of a function with bubbles, on the grid
        c("potential-129", "potential", (32, 32, 32), 5, 0.15, atoms=10, blmax=4, **T40),
        # forward and backward of the learned preconditioner on one sample
        c("train-129", "train", (32, 32, 32), 5, 0.15),
    ]


def draw(rng):
    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def cells(n_lo, n_hi, nlip, multiple=1):
        """Cells per axis of a box near n^3 points, sides up to 1.5 apart."""
        n = log_uniform(n_lo, n_hi)
        out = []
        for _ in range(3):
            side = min(n_hi, max(n_lo, n * rng.uniform(0.8, 1.2)))
            out.append(max(multiple, round((side - 1) / (nlip - 1) / multiple) * multiple))
        return out

    kind = rng.choice(["apply", "apply", "host", "batch", "batch", "gbfmm", "inject", "product",
                       "potential", "scf", "train"])
    nlip = rng.choice([5, 7])
    h = round(rng.uniform(0.1, 0.3), 4)
    quad = rng.choice([T18, T40, T50])
    energy = rng.choice([0.0, -round(log_uniform(0.05, 3.0), 4)])
    if kind == "apply":
        prec = rng.choice(["fp64", "fp64", "bf16x6", "bf16x3"])
        return _grid_case(kind, cells(21, 241, nlip), nlip, h, energy=energy, precision=prec,
                          **quad)
    if kind == "host":
        return _grid_case(kind, cells(21, 129, nlip), nlip, h, energy=energy, precision="fp64",
                          **quad)
    if kind == "batch":
        top, parts, points = log_uniform(33, 257), [], 0
        for _ in range(rng.randint(1, 4)):
            n = round((top * rng.uniform(0.5, 1.0)) / (nlip - 1)) * (nlip - 1) + 1
            k = min(rng.randint(1, 12), max(1, (120_000_000 - points) // n ** 3))
            points += k * n ** 3
            parts.append(f"{n}x{k}")
        return _grid_case(kind, (0, 0, 0), nlip, round(min(h, 0.2), 4), sizes=",".join(parts),
                          **T40)
    if kind == "gbfmm":
        boxes = rng.choice([2, 2, 3])
        return _grid_case(kind, cells(65, 225, nlip, 1 << boxes), nlip, round(min(h, 0.15), 4),
                          energy=rng.choice([0.0, 0.0, -0.6]), boxes=boxes,
                          lmax=rng.choice([6, 8, 12]), atoms=rng.randint(1, 8), blmax=4, **T50)
    if kind == "inject":
        return _grid_case(kind, cells(33, 257, nlip), nlip, h, atoms=rng.randint(1, 16),
                          blmax=rng.randint(0, 8))
    if kind == "product":
        return _grid_case(kind, cells(49, 129, nlip), nlip, h, atoms=rng.randint(2, 10),
                          blmax=rng.randint(1, 4))
    if kind == "potential":
        return _grid_case(kind, cells(33, 129, nlip), nlip, h, atoms=rng.randint(1, 10),
                          blmax=rng.randint(0, 4), **T40)
    if kind == "scf":
        return _grid_case(kind, cells(49, 129, 5), 5, h, orbitals=rng.randint(1, 14), **T40)
    return _grid_case("train", cells(17, 129, nlip), nlip, h)


def _shape(case):
    return tuple(case[a] * (case["nlip"] - 1) + 1 for a in ("cx", "cy", "cz"))


def _sizes(case):
    out = []
    for part in case["sizes"].split(","):
        n, k = part.split("x")
        out += [int(n)] * int(k)
    return out


# -------------------------------------------------------------- device views
class _Memory:
    """Device memory of the library as torch sees it; holds its owner."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 3}


def _view(owner, ptr, shape, typestr="<f8"):
    return torch.as_tensor(_Memory(owner, ptr, shape, typestr), device="cuda")


def _cube_view(cube):
    """(nz, ny, nx) view of a DeviceCube (x fastest)."""
    return _view(cube, cube.ptr, cube.shape[::-1])


_context = None


def _ctx():
    global _context
    if _context is None:
        _context = dage_amd.Context(0)
    return _context


# -------------------------------------------------------------------- inputs
def _axis(n, h, device="cuda"):
    return (torch.arange(n, dtype=torch.float64, device=device) - 0.5 * (n - 1)) * h


def _axes(shape, h):
    return [_axis(n, h) for n in shape]


def _gaussians(rng, axes, count, signed=False):
    """Sum of normalised Gaussians within the inner half of the box, as
    densities and orbital products are: (nz, ny, nx)."""
    x, y, z = axes
    q = rng.uniform(-1.0, 1.0, count) if signed else np.ones(count)
    alpha = np.exp(rng.uniform(np.log(0.3), np.log(5.0), count))
    cen = [rng.uniform(-0.5, 0.5, count) * float(a[-1]) for a in axes]
    t = functools.partial(torch.tensor, dtype=torch.float64, device="cuda")
    f = [torch.exp(-t(alpha)[:, None] * (a[None, :] - t(c)[:, None]) ** 2)
         for a, c in zip(axes, cen)]
    f[0] = f[0] * t(q * (alpha / math.pi) ** 1.5)[:, None]
    out = torch.zeros(len(z), len(y), len(x), dtype=torch.float64, device="cuda")
    for i in range(count):
        out += f[2][i][:, None, None] * (f[1][i][:, None] * f[0][i][None, :])
    return out


def _atoms(rng, case):
    """Charges, positions (at least 1.8 bohr apart where the box allows) and
    radial functions c_lm r^l exp(-Z r) (1 + O(r)) of each atom's bubbles."""
    shape = _shape(case)
    half = [0.4 * (n - 1) * case["h"] for n in shape]
    near, cen = 1.8, []
    while len(cen) < case["atoms"]:
        p = [rng.uniform(-a, a) for a in half]
        if all(math.dist(p, q) >= near for q in cen):
            cen.append(p)
        else:
            near *= 0.97
    charge = rng.choice([1.0, 6.0, 7.0, 8.0], case["atoms"])
    nlm = (case["blmax"] + 1) ** 2
    atoms = []
    for z, c in zip(charge, cen):
        steps = _radial_steps(z, 33, 7, 20.0)
        r = _radial_points(steps)
        coef = rng.uniform(-1.0, 1.0, (2, nlm))
        bf = np.zeros((len(r), nlm), order="F")
        for l in range(case["blmax"] + 1):
            for lm in range(l * l, (l + 1) * (l + 1)):
                bf[:, lm] = (coef[0, lm] + 0.2 * coef[1, lm] * r) * r ** l * np.exp(-z * r)
        atoms.append((np.array(c), float(z), steps, bf))
    return atoms


def _radial_steps(z, ncell, nlip, r_max):
    c = 8.0 * z ** -1.5
    edge = [0.0] + [c / ((r_max + c) / (i * (r_max / ncell)) - 1.0) for i in range(1, ncell + 1)]
    return np.diff(np.array(edge)) / (nlip - 1)


def _radial_points(steps, nlip=7):
    start = np.concatenate([[0.0], np.cumsum(steps * (nlip - 1))])
    pts = (start[:-1, None] + steps[:, None] * np.arange(nlip - 1)).ravel()
    return np.append(pts, start[-1])


def _bubbles(atoms, lmax, bfs=None):
    b = dage_amd.Bubbles(_ctx(), len(atoms), lmax, 0, 7)
    for i, (c, z, steps, bf) in enumerate(atoms):
        b.set_bubble(i, c, z, steps, bf if bfs is None else bfs[i])
    return b


def _second_bf(atoms, seed):
    """Another orbital's radial functions on the same atoms."""
    rng = np.random.default_rng([seed, 77])
    return [np.asfortranarray(bf * rng.uniform(-1.0, 1.0, bf.shape[1])[None, :])
            for _, _, _, bf in atoms]


def _grid(shape, nlip, h):
    return dage_amd.Grid3D(_ctx(), [-0.5 * (n - 1) * h for n in shape],
                           [np.full((n - 1) // (nlip - 1), h) for n in shape], nlip)


def _gauss(case):
    return dage_amd.GaussQuad(case["nlin"], case["nlog"], 2.0, case["tlog"])


def _cube(values):
    """A DeviceCube holding the (nz, ny, nx) tensor."""
    c = dage_amd.DeviceCube(_ctx(), tuple(values.shape[::-1]))
    _ctx().synchronize()
    _cube_view(c).copy_(values)
    return c


def _inputs(case, seed):
    """The numbers a case starts from, made from the seed alone."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "batch":
        sizes = _sizes(case)
        return {"rhs": [_gaussians(rng, _axes((n,) * 3, case["h"]), 4, True) for n in sizes],
                "energies": -0.5 * rng.uniform(0.1, 4.0, len(sizes))}
    axes = _axes(_shape(case), case["h"])
    if kind in ("apply", "host"):
        return {"rho": _gaussians(rng, axes, 8)}
    if kind == "gbfmm":
        return {"rho": _gaussians(rng, axes, 16), "atoms": _atoms(rng, case)}
    if kind == "inject":
        return {"atoms": _atoms(rng, case)}
    if kind == "product":
        return {"f": _gaussians(rng, axes, 6, True), "g": _gaussians(rng, axes, 6, True),
                "atoms": _atoms(rng, case)}
    if kind == "potential":
        return {"rho": _gaussians(rng, axes, 6, True), "atoms": _atoms(rng, case)}
    if kind == "scf":
        vnuc = -sum(float(z) * _smeared(axes, p) for z, p in
                    zip(rng.choice([1.0, 6.0, 7.0, 8.0], 6),
                        rng.uniform(-0.4, 0.4, (6, 3)) * [float(a[-1]) for a in axes]))
        return {"vnuc": vnuc,
                "psi": [_gaussians(rng, axes, 3, True) for _ in range(case["orbitals"])],
                "eps": np.sort(-0.5 * rng.uniform(0.2, 4.0, case["orbitals"]))}
    shape = tuple(n for n in _shape(case)[::-1])
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    psi = _gaussians(rng, axes, 4, True)
    delta = _gaussians(rng, axes, 4, True)
    x = torch.stack([psi, delta / delta.square().mean().sqrt()]).float()
    t = torch.randn(shape, generator=g, device="cuda") * 0.1 + x[1]
    w = []
    for ci, co in learned.LAYERS:
        w.append((rng.standard_normal((co, ci, 27)).astype(np.float32) * math.sqrt(2 / (27 * ci)),
                  0.05 * rng.standard_normal(co).astype(np.float32)))
    return {"x": x, "t": t, "w": w}


def _smeared(axes, p):
    x, y, z = axes
    r = torch.sqrt((x[None, None, :] - p[0]) ** 2 + (y[None, :, None] - p[1]) ** 2
                   + (z[:, None, None] - p[2]) ** 2).clamp_min(1e-9)
    return torch.erf(2.0 * r) / r


# ------------------------------------------------------------ prepare and run
def prepare(case, seed):
    kind, ctx, v = case["kind"], _ctx(), _inputs(case, seed)
    s = {"case": case}
    if kind == "batch":
        sizes = _sizes(case)
        grids = {n: _grid((n,) * 3, case["nlip"], case["h"]) for n in sizes}
        b = dage_amd.HelmholtzBatch(ctx, [grids[n] for n in sizes], v["energies"], _gauss(case))
        ctx.synchronize()
        for i, rhs in enumerate(v["rhs"]):
            _view(b, b.input_ptr(i), rhs.shape).copy_(rhs)
        s.update(batch=b, grids=grids, energies=v["energies"],
                 out=[_view(b, b.output_ptr(i), rhs.shape) for i, rhs in enumerate(v["rhs"])])
        torch.cuda.synchronize()
        return s
    shape = _shape(case)
    grid = s["grid"] = _grid(shape, case["nlip"], case["h"])
    if kind in ("apply", "host"):
        op = dage_amd.Helmholtz3D(ctx, grid, grid, _gauss(case), energy=case["energy"])
        s["op"] = op
        if kind == "host":
            s["rho"] = np.asfortranarray(v["rho"].cpu().numpy().transpose(2, 1, 0))
        else:
            s["rho"], s["out"] = _cube(v["rho"]), dage_amd.DeviceCube(ctx, shape)
    elif kind == "gbfmm":
        fmm = dage_amd.GBFMMCoulomb3D(ctx, grid, maxlevel=case["boxes"], lmax=case["lmax"],
                                      gauss=_gauss(case))
        if case["energy"] != 0.0:
            fmm.set_energy(case["energy"])
        s.update(fmm=fmm, bub=_bubbles(v["atoms"], case["blmax"]), rho=_cube(v["rho"]),
                 total=dage_amd.DeviceCube(ctx, shape), pot=dage_amd.DeviceCube(ctx, shape))
    elif kind == "inject":
        s.update(bub=_bubbles(v["atoms"], case["blmax"]), out=dage_amd.DeviceCube(ctx, shape))
    elif kind == "product":
        bf2 = _second_bf(v["atoms"], seed)
        for key, bfs in (("f", None), ("g", bf2)):
            s[key] = f3d.Function3D(grid, _cube(v[key]), _bubbles(v["atoms"], case["blmax"], bfs),
                                    type=f3d.F3D_TYPE_CUSP)
    elif kind == "potential":
        s["op"] = dage_amd.Coulomb3D(ctx, grid, grid, _gauss(case))
        s["f"] = f3d.Function3D(grid, _cube(v["rho"]), _bubbles(v["atoms"], case["blmax"]),
                                type=f3d.F3D_TYPE_CUSP)
    elif kind == "scf":
        mol = scf.Molecule(np.zeros(0), np.zeros((0, 3)))
        S = scf.HelmholtzSCF(ctx, grid, mol, case["orbitals"], gauss=_gauss(case),
                             external_potential=v["vnuc"].cpu().numpy().transpose(2, 1, 0))
        ctx.synchronize()
        for p, psi in zip(S.psi, v["psi"]):
            _cube_view(p).copy_(psi)
        S.eps[:] = v["eps"]
        s["scf"] = S
    else:
        m = learned.ConvPreconditioner(ctx, shape)
        m.set_weights(v["w"])
        ctx.synchronize()
        _view(m, m.act[0].ptr, v["x"].shape, "<f4").copy_(v["x"])
        s.update(model=m, t=v["t"])
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "batch":
        s["batch"].set_energies(s["energies"])
        s["batch"].apply()
        return s["out"]
    if kind == "apply":
        s["op"].transform_cuda_cube(s["rho"], s["out"], PREC[case["precision"]])
        return _cube_view(s["out"])
    if kind == "host":
        s["op"].set_energy(case["energy"])
        return s["op"].transform_cube(s["rho"])
    if kind == "gbfmm":
        s["total"].copy_from(s["rho"])
        s["bub"].inject(s["grid"], s["total"])
        s["fmm"].apply_device(s["total"], s["pot"])
        return [_cube_view(s["total"]), _cube_view(s["pot"])]
    if kind == "inject":
        s["out"].set_to_zero()
        s["bub"].inject(s["grid"], s["out"])
        return _cube_view(s["out"])
    if kind == "product":
        p = s["f"].multiply(s["g"])
        value = p.integrate()
        p.bubbles.close()
        return [_cube_view(p.cube), value]
    if kind == "potential":
        p = f3d.operate_on(s["op"], s["f"])
        p.bubbles.inject(s["grid"], p.cube)
        return _cube_view(p.cube)
    if kind == "scf":
        S = s["scf"]
        S.build_potential()
        S.helmholtz_step()
        eps, _, kinetic = S.ritz(S.psi)
        return [_cube_view(S.V), [_cube_view(d) for d in S.delta], eps, kinetic]
    m, nx, ny, nz = s["model"], *_shape(case)
    m.forward()
    loss = ctypes.c_double()
    call("dage_mse_loss", m.ctx.handle, m.vol, ctypes.c_void_p(m.act[-1].ptr),
         ctypes.c_void_p(s["t"].data_ptr()), ctypes.c_void_p(m.grad[3].ptr), ctypes.byref(loss))
    m.backward()
    return [loss.value, _view(m, m.act[-1].ptr, (nz, ny, nx), "<f4"),
            [[_view(m, P["gw"].ptr, (P["co"], P["ci"], 27), "<f4"),
              _view(m, P["gb"].ptr, (P["co"],), "<f4")] for P in m.params]]


# -------------------------------------------------------------- work, tolerance
def _tensor_flops(shape, T):
    return 6.0 * T * float(np.prod(shape)) * sum(shape) / 3.0


def work(case):
    """Inputs read once and outputs written once; FLOPs of the tensor form
    (three dense mode products per t-point) and of the point-wise sums."""
    kind = case["kind"]
    if kind == "batch":
        sizes, T = _sizes(case), case["nlin"] + case["nlog"]
        return {"bytes": 16.0 * sum(n ** 3 for n in sizes),
                "flops": sum(_tensor_flops((n,) * 3, T) for n in sizes)}
    shape, pts = _shape(case), float(np.prod(_shape(case)))
    T = case.get("nlin", 0) + case.get("nlog", 0)
    # per point and bubble: Horner polynomials, radial dot products, harmonics
    nlm = (case.get("blmax", 0) + 1) ** 2
    inject = pts * case.get("atoms", 0) * (98.0 + 20.0 * nlm)
    if kind in ("apply", "host"):
        return {"bytes": 16.0 * pts, "flops": _tensor_flops(shape, T)}
    if kind == "gbfmm":
        return {"bytes": 24.0 * pts, "flops": inject + _tensor_flops(shape, T)}
    if kind == "inject":
        return {"bytes": 8.0 * pts, "flops": inject}
    if kind == "product":
        n12 = (2 * max(case["blmax"], 2) + 1) ** 2
        return {"bytes": 24.0 * pts,
                "flops": 2 * inject + pts * case["atoms"] * (98.0 + 20.0 * n12)}
    if kind == "potential":
        return {"bytes": 16.0 * pts, "flops": inject + _tensor_flops(shape, T)}
    if kind == "scf":
        k = case["orbitals"]
        return {"bytes": (2 * k + 2) * 8.0 * pts,
                "flops": (k + 1) * _tensor_flops(shape, T) + 6.0 * k * k * pts}
    macs = sum(27.0 * ci * co for ci, co in learned.LAYERS)
    first = 27.0 * learned.LAYERS[0][0] * learned.LAYERS[0][1]
    return {"bytes": 4.0 * 4 * pts, "flops": 2.0 * pts * (3.0 * macs - first)}


def tolerance(case):
    """About four times the distance from exact() (2-norm): 3e-8 for bf16x6,
    1e-6 for bf16x3, 6e-6 for the FP32 filter gradients, 1e-14 where bubbles
    are only summed.  The operators' matrix entries come from closed forms
    that cancel: 2.5e-11 of the potential on odd boxes."""
    prec = case.get("precision", "fp64")
    if prec != "fp64":
        return {"rel": 1.2e-7 if prec == "bf16x6" else 4e-6}
    return {"train": {"rel": 2.5e-5}, "inject": {"rel": 3e-14, "max": 3e-12},
            "product": {"rel": 4e-14, "max": 3e-12}}.get(case["kind"], {"rel": 1e-10})


# --------------------------------------------------------------------- exact
def exact(case, seed):
    kind, v = case["kind"], _inputs(case, seed)
    if kind == "batch":
        out = []
        for n, rhs, e in zip(_sizes(case), v["rhs"], v["energies"]):
            out.append(_exact_apply(case, (n,) * 3, rhs, e, True))
        return out
    shape = _shape(case)
    axes = _axes(shape, case["h"])
    if kind in ("apply", "host"):
        out = _exact_apply(case, shape, v["rho"], case["energy"], True)
        return out.permute(2, 1, 0).cpu().numpy() if kind == "host" else out
    if kind == "gbfmm":
        # the potential without the expansions' truncation (about 1e-5)
        total = v["rho"] + _exact_inject(axes, _bubble_tables(v["atoms"]))
        return [total, _exact_apply(case, shape, total, case["energy"], False)]
    if kind == "inject":
        return _exact_inject(axes, _bubble_tables(v["atoms"]))
    if kind == "product":
        return _exact_product(case, seed, axes, v)
    if kind == "potential":
        tables = _bubble_tables(v["atoms"])
        pots = [(c, steps, _exact_radial_coulomb(steps, bf)) for c, steps, bf in tables]
        return (_exact_apply(case, shape, v["rho"], 0.0, True) + _exact_inject(axes, pots))
    if kind == "scf":
        return _exact_scf(case, shape, v)
    return _exact_train(v)


def _exact_quad(case):
    """Gauss-Legendre points and weights: linear on [0, 2], logarithmic above."""
    x, w = np.polynomial.legendre.leggauss(case["nlin"])
    t0, w0 = x + 1.0, w
    x, w = np.polynomial.legendre.leggauss(case["nlog"])
    ratio = case["tlog"] / 2.0
    t1 = 2.0 * ratio ** (0.5 * (x + 1.0))
    return np.concatenate([t0, t1]), np.concatenate([w0, 0.5 * math.log(ratio) * w * t1])


def _lagrange(nlip):
    """Coefficients (node, power) of the nlip Lagrange polynomials on 0..nlip-1."""
    c = np.zeros((nlip, nlip))
    for j in range(nlip):
        p = np.array([1.0])
        for m in range(nlip):
            if m != j:
                p = np.convolve(p, [-float(m), 1.0][::-1]) / (j - m)
        c[j] = p[::-1]
    return c


def _basis(nlip, u):
    """Values of the Lagrange polynomials at u (any shape): (..., nlip)."""
    k = torch.arange(nlip, dtype=torch.float64, device=u.device)
    out = torch.ones(*u.shape, nlip, dtype=torch.float64, device=u.device)
    for j in range(nlip):
        for m in range(nlip):
            if m != j:
                out[..., j] *= (u - k[m]) / (j - m)
    return out


def _exact_matrix(n, nlip, h, t):
    """F(o, i) = integral of exp(-t^2 (x_o - x)^2) times the i-th cell basis
    function, each cell cut at x_o and at 7.2 widths from it, 40 points each."""
    x = _axis(n, h)
    ncell = (n - 1) // (nlip - 1)
    a = x[:: nlip - 1][:ncell]
    b = a + (nlip - 1) * h
    gx, gw = np.polynomial.legendre.leggauss(40)
    gx, gw = (torch.tensor(g, dtype=torch.float64, device="cuda") for g in (gx, gw))
    F = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    cut = 7.2 / t
    for lo, hi in ((x - cut, x), (x, x + cut)):
        l = torch.maximum(a[None, :], lo[:, None])
        r = torch.minimum(b[None, :], hi[:, None])
        half = 0.5 * (r - l).clamp_min(0.0)
        xs = (0.5 * (l + r))[..., None] + half[..., None] * gx
        g = torch.exp(-(t * (x[:, None, None] - xs)) ** 2) * gw * half[..., None]
        part = torch.einsum("ocq,ocqj->ocj", g, _basis(nlip, (xs - a[None, :, None]) / h))
        for j in range(nlip):
            F[:, j: j + (ncell - 1) * (nlip - 1) + 1: nlip - 1] += part[:, :, j]
    return F


def _exact_apply(case, shape, rho, energy, coda):
    tp, tw = _exact_quad(case)
    out = torch.zeros_like(rho)
    for t, w in zip(tp, tw):
        F = {n: _exact_matrix(n, case["nlip"], case["h"], float(t)) for n in set(shape)}
        w = 2.0 / math.sqrt(math.pi) * w
        if energy < -0.005:
            w *= math.exp(2.0 * energy / (4.0 * t * t))
        nx, ny, nz = shape
        u = (rho.reshape(-1, nx) @ F[nx].t()).reshape(nz, ny, nx)
        u = torch.stack([F[ny] @ plane for plane in u])
        out += w * (F[nz] @ u.reshape(nz, -1)).reshape(nz, ny, nx)
    return out + (math.pi / case["tlog"] ** 2) * rho if coda else out


def _bubble_tables(atoms, bfs=None):
    return [(c, steps, bf if bfs is None else bfs[i]) for i, (c, _, steps, bf) in enumerate(atoms)]


def _harmonics(lmax, x, y, z):
    """Racah real solid harmonics, m from -l to l for each l."""
    S = [torch.ones_like(x)]
    if lmax >= 1:
        S += [y, z, x]
    r2 = x * x + y * y + z * z
    for l in range(2, lmax + 1):
        p, q = (l - 1) ** 2 + l - 1, (l - 2) ** 2 + l - 2
        f = math.sqrt((2 * l - 1) / (2 * l))
        row = [f * (y * S[p + l - 1] + x * S[p - l + 1])]
        for m in range(-l + 1, l):
            u = (2 * l - 1) / math.sqrt((l + m) * (l - m)) * z * S[p + m]
            if l - abs(m) > 1:
                u = u - math.sqrt((l + m - 1) * (l - m - 1) / ((l + m) * (l - m))) * r2 * S[q + m]
            row.append(u)
        row.append(f * (x * S[p + l - 1] - y * S[p - l + 1]))
        S += row
    return S


def _bubble_values(table, x, y, z):
    """One bubble at the points (flat tensors): sum of f_lm(r) S_lm / r^l."""
    c, steps, bf = table
    dev = x.device
    lmax = math.isqrt(bf.shape[1]) - 1
    st = torch.tensor(steps, dtype=torch.float64, device=dev)
    edge = torch.tensor(_radial_points(steps)[::6], dtype=torch.float64, device=dev)
    f = torch.tensor(np.ascontiguousarray(bf), dtype=torch.float64, device=dev)
    x, y, z = x - float(c[0]), y - float(c[1]), z - float(c[2])
    r = torch.sqrt(x * x + y * y + z * z)
    cell = (torch.searchsorted(edge, r.detach(), right=True) - 1).clamp(0, len(steps) - 1)
    inside = (r.detach() <= edge[-1]).to(torch.float64)
    u = (r - edge[cell]) / st[cell]
    k = torch.arange(7, dtype=torch.float64, device=dev)
    basis = []
    for j in range(7):
        p = torch.ones_like(u)
        for m in range(7):
            if m != j:
                p = p * (u - k[m]) / (j - m)
        basis.append(p)
    inv = torch.where(r > 0, 1.0 / r.clamp_min(1e-300), torch.ones_like(r))
    S = _harmonics(lmax, x * inv, y * inv, z * inv)
    out = torch.zeros_like(x)
    for lm in range(bf.shape[1]):
        col = f[:, lm].contiguous()
        out = out + S[lm] * sum(col[cell * 6 + j] * basis[j] for j in range(7))
    return out * inside


def _exact_inject(axes, tables):
    x, y, z = axes
    out = torch.zeros(len(z), len(y), len(x), dtype=torch.float64, device="cuda")
    chunk = max(1, 4_000_000 // (len(x) * len(y)))
    for k in range(0, len(z), chunk):
        zz, yy, xx = torch.meshgrid(z[k:k + chunk], y, x, indexing="ij")
        for t in tables:
            out[k:k + chunk] += _bubble_values(t, xx.reshape(-1), yy.reshape(-1),
                                               zz.reshape(-1)).reshape(xx.shape)
    return out


def _exact_radial_coulomb(steps, bf):
    """4 pi/(2l+1) [r^-(l+1) int_0^r s^(l+2) f + r^l int_r^R s^(1-l) f], the
    integrands interpolated cell by cell."""
    r = _radial_points(steps)
    c = _lagrange(7)
    anti = c / np.arange(1, 8)  # of u^(p+1)
    upto = np.array([[np.sum(anti[j] * m ** np.arange(1.0, 8.0)) for j in range(7)]
                     for m in range(7)])  # integral of L_j from 0 to m
    out = np.zeros_like(bf)
    with np.errstate(divide="ignore"):
        power = {n: np.where((r == 0) & (n < 0), 0.0, r ** float(n)) for n in
                 range(-math.isqrt(bf.shape[1]) - 1, math.isqrt(bf.shape[1]) + 3)}
    for l in range(math.isqrt(bf.shape[1])):
        for lm in range(l * l, (l + 1) ** 2):
            g = [bf[:, lm] * power[l + 2], bf[:, lm] * power[1 - l]]
            cum = []
            for f in g:
                cells = np.stack([f[6 * i:6 * i + 7] for i in range(len(steps))])
                part = (cells @ upto.T) * steps[:, None]  # from the cell's start to its node m
                start = np.concatenate([[0.0], np.cumsum(part[:, 6])])
                cum.append(np.append((start[:-1, None] + part[:, :6]).ravel(), start[-1]))
            inner, outer = cum[0], cum[1][-1] - cum[1]
            out[:, lm] = 4.0 * math.pi / (2 * l + 1) * (power[-l - 1] * inner + power[l] * outer)
    return out


def _sphere(lmax):
    """Directions, weights and harmonics of a rule exact for degree 2 lmax."""
    ct, w = np.polynomial.legendre.leggauss(lmax + 2)
    ph = 2.0 * math.pi * np.arange(2 * lmax + 3) / (2 * lmax + 3)
    st = np.sqrt(1.0 - ct ** 2)
    u = np.stack([(st[:, None] * np.cos(ph)).ravel(), (st[:, None] * np.sin(ph)).ravel(),
                  (ct[:, None] + 0 * ph).ravel()])
    wt = (w[:, None] * (2.0 * math.pi / len(ph)) + 0 * ph).ravel()
    S = torch.stack(_harmonics(lmax, *(torch.tensor(a) for a in u))).numpy()
    return u, wt, S


def _exact_product(case, seed, axes, v):
    """(cube + bubbles) (cube + bubbles) less the product bubbles
    B1 B2 + B1 T2 + T1 B2, T the second-order Taylor bubbles at each atom."""
    t1, t2 = _bubble_tables(v["atoms"]), _bubble_tables(v["atoms"], _second_bf(v["atoms"], seed))
    big = 2 * max(case["blmax"], 2)
    u, wt, S = _sphere(big)
    project = np.concatenate([S[l * l:(l + 1) ** 2] * wt * (2 * l + 1) / (4.0 * math.pi)
                              for l in range(big + 1)])
    taylor = [_taylor_parts(case, axes, v[key], tables) for key, tables in (("f", t1), ("g", t2))]
    prod, integral = [], 0.0
    for i, (c, steps, bf) in enumerate(t1):
        r = _radial_points(steps)
        n = bf.shape[1]
        with np.errstate(divide="ignore"):
            damp = np.array([1.0 if q <= 2.3e-16 else 0.5 * math.erfc(q - 2.0 / q) for q in r])
        B, T = [], []
        for tables, parts in ((t1, taylor[0]), (t2, taylor[1])):
            B.append(tables[i][2] @ S[:n])
            value, grad, hess = parts[i]
            # every Cartesian term of degree d carries 1/d!, so a mixed second
            # derivative counts once at 1/2
            quad = 0.5 * sum(hess[a, b] * u[a] * u[b] for a in range(3) for b in range(a, 3))
            T.append(damp[:, None] * (value + r[:, None] * (grad @ u) + r[:, None] ** 2 * quad))
        f = (B[0] * B[1] + B[0] * T[1] + T[0] * B[1]) @ project.T
        prod.append((c, steps, f))
        w = _radial_weights(steps)
        integral += 4.0 * math.pi * float(np.sum(w * r ** 2 * f[:, 0]))
    cube = ((v["f"] + _exact_inject(axes, t1)) * (v["g"] + _exact_inject(axes, t2))
            - _exact_inject(axes, prod))
    return [cube, integral + float(_weighted(case, cube).sum())]


def _radial_weights(steps):
    cell = np.array([np.sum(_lagrange(7)[j] * 6.0 ** np.arange(1.0, 8.0) / np.arange(1, 8))
                     for j in range(7)])
    w = np.zeros(6 * len(steps) + 1)
    for i, h in enumerate(steps):
        w[6 * i:6 * i + 7] += h * cell
    return w


def _line_weights(n, nlip, h):
    m = nlip - 1
    cell = np.array([np.sum(_lagrange(nlip)[j] * float(m) ** np.arange(1.0, nlip + 1.0)
                            / np.arange(1, nlip + 1)) for j in range(nlip)])
    w = np.zeros(n)
    for c in range((n - 1) // m):
        w[c * m:c * m + nlip] += h * cell
    return torch.tensor(w, device="cuda")


def _weighted(case, cube):
    wx, wy, wz = (_line_weights(n, case["nlip"], case["h"]) for n in cube.shape[::-1])
    return cube * wz[:, None, None] * wy[:, None] * wx


def _taylor_parts(case, axes, cube, tables):
    """Value, gradient and Hessian at every atom of the cube's interpolant plus
    the other atoms' bubbles."""
    nlip, h, cpu = case["nlip"], case["h"], cube.cpu()
    out = []
    for i, (c, _, _) in enumerate(tables):
        def at(p):
            total = torch.zeros((), dtype=torch.float64)
            blocks, basis = [], []
            for a in range(3):
                x0, n = float(axes[a][0]), len(axes[a])
                cell = min(max(int((float(c[a]) - x0) / (h * (nlip - 1))), 0),
                           (n - 1) // (nlip - 1) - 1)
                u = (p[a] - x0) / h - cell * (nlip - 1)
                row = []
                for j in range(nlip):
                    q = torch.ones((), dtype=torch.float64)
                    for m in range(nlip):
                        if m != j:
                            q = q * (u - m) / (j - m)
                    row.append(q)
                basis.append(torch.stack(row))
                blocks.append(slice(cell * (nlip - 1), cell * (nlip - 1) + nlip))
            total = total + torch.einsum("zyx,z,y,x->", cpu[blocks[2], blocks[1], blocks[0]],
                                         basis[2], basis[1], basis[0])
            for k, other in enumerate(tables):
                if k != i:
                    total = total + _bubble_values(other, p[0:1], p[1:2], p[2:3])[0]
            return total

        p = torch.tensor(c, dtype=torch.float64)
        grad = torch.autograd.functional.jacobian(at, p)
        hess = torch.autograd.functional.hessian(at, p)
        out.append((float(at(p)), grad.numpy(), hess.numpy()))
    return out


def _exact_scf(case, shape, v):
    rho = 2.0 * sum(p * p for p in v["psi"])
    V = v["vnuc"] + _exact_apply(case, shape, rho, 0.0, True)
    V = V - (3.0 / math.pi) ** (1.0 / 3.0) * rho.clamp_min(0.0) ** (1.0 / 3.0)
    deltas = [-_exact_apply(case, shape, V * p, float(e), True) / (2.0 * math.pi) - p
              for p, e in zip(v["psi"], v["eps"])]
    k, nlip, h = case["orbitals"], case["nlip"], case["h"]
    wts = [_line_weights(n, nlip, h) for n in shape]
    flat = torch.stack([p.reshape(-1) for p in v["psi"]])
    full = (wts[2][:, None, None] * wts[1][:, None] * wts[0]).reshape(-1)
    S = (flat * full) @ flat.t()
    T = torch.zeros(k, k, dtype=torch.float64, device="cuda")
    for a in range(3):  # grid axis a is tensor axis 2 - a
        K = _stiffness(shape[a], nlip, h) / wts[a][:, None]
        kf = torch.stack([torch.movedim(torch.tensordot(K, p, dims=([1], [2 - a])), 0, 2 - a)
                          .reshape(-1) for p in v["psi"]])
        T += 0.5 * (flat * full) @ kf.t()
    H = T + (flat * full) @ (flat * V.reshape(-1)).t()
    H, S = (0.5 * (m + m.t()).cpu().numpy() for m in (H, S))
    s, U = np.linalg.eigh(S)
    keep = s > 1e-10 * s[-1]
    X = U[:, keep] / np.sqrt(s[keep])
    return [V, deltas, np.linalg.eigvalsh(X.T @ H @ X), T.cpu().numpy()]


def _stiffness(n, nlip, h):
    c = _lagrange(nlip)
    d = c[:, 1:] * np.arange(1, nlip)
    m = float(nlip - 1)
    Kc = np.array([[sum(d[a, p] * d[b, q] * m ** (p + q + 1) / (p + q + 1)
                        for p in range(nlip - 1) for q in range(nlip - 1))
                    for b in range(nlip)] for a in range(nlip)]) / h
    K = np.zeros((n, n))
    for cell in range((n - 1) // (nlip - 1)):
        s = slice(cell * (nlip - 1), cell * (nlip - 1) + nlip)
        K[s, s] += Kc
    return torch.tensor(K, device="cuda")


def _exact_train(v):
    """The network in 64 bits on the bf16-rounded weights: loss, output and
    the gradients by hand-written backward passes."""
    nz, ny, nx = v["t"].shape
    pad = torch.nn.functional.pad

    def windows(a):
        p = pad(a, (1, 1, 1, 1, 1, 1))
        for t in range(27):
            dx, dy, dz = t % 3, (t // 3) % 3, t // 9
            yield t, p[:, dz:dz + nz, dy:dy + ny, dx:dx + nx].reshape(a.shape[0], -1)

    def conv(a, w):
        out = torch.zeros(w.shape[0], nz * ny * nx, dtype=torch.float64, device="cuda")
        for t, win in windows(a):
            out += w[:, :, t] @ win
        return out.reshape(-1, nz, ny, nx)

    ws = [(torch.tensor(w, device="cuda").bfloat16().double(),
           torch.tensor(b, device="cuda").double()) for w, b in v["w"]]
    acts = [v["x"].double()]
    for i, (w, b) in enumerate(ws):
        a = conv(acts[-1], w) + b[:, None, None, None]
        acts.append(a.clamp_min(0.0) if i < len(ws) - 1 else a)
    diff = acts[-1][0] - v["t"].double()
    g = (2.0 / diff.numel()) * diff[None]
    grads = [None] * len(ws)
    for i in range(len(ws) - 1, -1, -1):
        flat = g.reshape(g.shape[0], -1)
        gw = torch.stack([flat @ win.t() for _, win in windows(acts[i])], dim=2)
        grads[i] = [gw.float(), flat.sum(1).float()]
        if i:
            g = conv(g, ws[i][0].transpose(0, 1).flip(2).contiguous()) * (acts[i] > 0)
    return [float(diff.square().mean()), acts[-1][0].float(), grads]
