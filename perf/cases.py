"""What a user of this framework has it do, as cases that can be timed.

A case is one call (or one forward and backward pair) of a public entry point
on inputs made from a seed:

  project   ``MacPlan.project``: the MAC projection on per-box arrays, planar
            beta0 in 2D and 3D or a star's beta0 on the faces, device arrays or
            (``host``) the numpy arrays a Fortran caller's MultiFabs amount to
  twolevel  ``MacMLPlan.project``: a coarse level and one refined region
  diffuse   ``MacPlan.solve``: thermal diffusion, (alpha - D beta G) phi = rh
  gradient  ``autograd.mac_project`` forward, and backward through a loss
  inputs    ``make_macrhs`` and ``make_s0mac`` on a star's geometry

Domains are boxes of cubic cells, extents multiples of 16 (MAESTRO's blocking
factors), chopped into boxes of at most ``box`` cells a side.  Per-box arrays
are views into one buffer per quantity, as an arena allocator lays a MultiFab
out, each on a 512-byte boundary.  A call updates its velocities and its
pressure in place, so ``run`` first brings the unprojected velocities and a
zero guess back, which stands for the advection step that makes new ones.
"""
import math

import numpy as np
import torch

from maestro_amd import autograd, mac

PER, WALL, OUT = mac.PERIODIC, mac.SLIP_WALL, mac.OUTLET
PREC = {"fp64": mac.PREC_FP64, "mixed": mac.PREC_MIXED, "bf16": mac.PREC_MIXED_BF16}


def listed():
    P = dict(kind="project", beta0="planar", omega=0.0, top="wall", macrhs=False, host=False)
    return [
        # the smallest call: a 2D convection test problem, the library's default options
        {**P, "name": "plane2_128_fp64", "nx": 128, "ny": 128, "nz": 1, "box": 32, "precision": "fp64"},
        # a 2D atmosphere of ragged extents, open at the top, with the divergence constraint's source
        {**P, "name": "plane2_640x384_mixed", "nx": 640, "ny": 384, "nz": 1, "box": 64, "precision": "mixed",
         "top": "outlet", "macrhs": True},
        # the drop-in as a Fortran host calls it: host arrays, default options, a small 3D domain
        {**P, "name": "plane3_64_host_fp64", "nx": 64, "ny": 64, "nz": 64, "box": 32, "precision": "fp64",
         "host": True, "macrhs": True},
        # ragged 3D boxes, open at the top, the reference's algorithm
        {**P, "name": "plane3_96x80x112_fp64", "nx": 96, "ny": 80, "nz": 112, "box": 32, "precision": "fp64",
         "top": "outlet", "macrhs": True},
        # an ordinary plane-parallel run per GPU
        {**P, "name": "plane3_128_mixed", "nx": 128, "ny": 128, "nz": 128, "box": 64, "precision": "mixed"},
        # the headline workload: 256^3, mixed precision with over-relaxed sweeps
        {**P, "name": "plane3_256_mixed_sor", "nx": 256, "ny": 256, "nz": 256, "box": 64, "precision": "mixed",
         "omega": 1.25},
        # the same workload with the reference's algorithm throughout
        {**P, "name": "plane3_256_fp64", "nx": 256, "ny": 256, "nz": 256, "box": 64, "precision": "fp64"},
        # the largest: a spherical star, beta0 on the faces, outflow on every side
        {**P, "name": "star_512_mixed", "nx": 512, "ny": 512, "nz": 512, "box": 64, "precision": "mixed",
         "beta0": "star", "top": "outlet"},
        # adaptive mesh: two levels, the refined region on the bottom wall
        {"name": "twolevel_128_fp64", "kind": "twolevel", "nx": 128, "ny": 128, "nz": 128, "box": 32,
         "rx": 32, "ry": 32, "rz": 0, "mx": 64, "my": 64, "mz": 64, "precision": "fp64"},
        # a thermal diffusion step on an extent that is no power of two
        {"name": "diffuse_192_mixed", "kind": "diffuse", "nx": 192, "ny": 192, "nz": 192, "box": 64,
         "precision": "mixed"},
        # gradients through the projection: forward, then backward
        {"name": "gradient_128_mixed", "kind": "gradient", "nx": 128, "ny": 128, "nz": 128, "precision": "mixed"},
        # the producers of a star's inputs
        {"name": "inputs_256", "kind": "inputs", "nx": 256, "ny": 256, "nz": 256, "box": 64},
    ]


def _extent(rng, lo, hi):
    """A multiple of 16 between lo and hi, spread over the logarithm; a
    multiple of 32 above 128 (the multigrid's bottom level stays small)."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    q = 16 if v <= 128 else 32
    return int(min(hi, max(lo, q * round(v / q))))


def _extents(rng, lo, hi, most):
    while True:
        n = [_extent(rng, lo, hi) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most and max(n) <= 6 * min(n):
            return n


def draw(rng):
    kind = rng.choice(["plane3"] * 6 + ["plane2"] * 3 + ["star"] * 2 + ["twolevel"] * 2 + ["diffuse"] * 2 +
                      ["gradient"] * 2 + ["host", "inputs"])
    prec = rng.choice(["fp64", "mixed", "mixed", "bf16"])
    box = rng.choice([32, 48, 64])
    if kind in ("plane3", "plane2", "star", "host"):
        c = dict(kind="project", beta0="planar", omega=rng.choice([0.0, 0.0, 1.25]), top=rng.choice(["wall", "outlet"]),
                 macrhs=rng.random() < 0.5, host=kind == "host", precision=prec, box=box)
        if kind == "plane2":
            while True:
                n = [_extent(rng, 64, 1024), _extent(rng, 64, 1024), 1]
                if max(n[:2]) <= 6 * min(n[:2]):
                    break
        elif kind == "host":
            n = _extents(rng, 32, 128, 128 ** 3)
        else:
            n = _extents(rng, 32, 320, 256 ** 3)
        if kind == "star":
            c.update(beta0="star", top="outlet", macrhs=False)
        return {**c, "nx": n[0], "ny": n[1], "nz": n[2]}
    if kind == "twolevel":
        n = _extents(rng, 48, 128, 128 ** 3)
        # the refined rectangle, in coarse cells: multiples of 8, off the domain's sides except the bottom
        m = [8 * rng.randint(2, max(2, n[d] // 16)) for d in range(3)]
        r = [8 * rng.randint(1, (n[d] - m[d]) // 8 - 1) for d in range(2)] + [0]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "box": 32, "rx": r[0], "ry": r[1], "rz": r[2],
                "mx": m[0], "my": m[1], "mz": m[2], "precision": rng.choice(["fp64", "mixed"])}
    n = _extents(rng, 32, 320, 256 ** 3)
    c = {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2]}
    if kind == "diffuse":
        return {**c, "box": box, "precision": rng.choice(["fp64", "mixed"])}
    if kind == "gradient":
        return {**c, "precision": rng.choice(["fp64", "mixed"])}
    return {**c, "box": box}


# ------------------------------------------------------------------ layouts
def _cuts(n, most):
    """[lo, hi] of the pieces of n cells, at most ``most`` each, multiples of 8 where n is one."""
    pieces = -(-n // most)
    unit = 8 if n % 8 == 0 else 1
    q, r = divmod(n // unit, pieces)
    out, lo = [], 0
    for p in range(pieces):
        w = unit * (q + (p < r))
        out.append((lo, lo + w - 1))
        lo += w
    return out


def _boxes(n, most):
    dim = 3 if n[2] > 1 else 2
    cx, cy = _cuts(n[0], most), _cuts(n[1], most)
    cz = _cuts(n[2], most) if dim == 3 else [(0, 0)]
    return [((x[0], y[0], z[0]), (x[1], y[1], z[1])) for z in cz for y in cy for x in cx]


def _ext(case):
    return (case["nx"], case["ny"], case["nz"])


def _bc(case):
    """Physical boundary codes: x and y periodic, a wall below, ``top`` above; a star is open on every side."""
    dim = 3 if case["nz"] > 1 else 2
    if case.get("beta0") == "star":
        return [[OUT, OUT]] * 3
    return [[PER, PER]] * (dim - 1) + [[WALL, OUT if case.get("top") == "outlet" else WALL]]


class Arena:
    """One buffer holding the per-box arrays of one quantity: box b, face
    direction d (or -1 for cells) with ng ghost layers."""

    def __init__(self, boxes, dim, dirs, ng, host=False):
        self.boxes, self.dim, self.dirs, self.ng, self.host = boxes, dim, dirs, ng, host
        self.shapes, self.offs, total = [], [], 0
        for lo, hi in boxes:
            for d in dirs:
                shp = tuple(hi[e] - lo[e] + 1 + ((2 * ng + (e == d)) if e < dim else 0) for e in (2, 1, 0))
                self.shapes.append(shp)
                self.offs.append(total)
                total += -(-math.prod(shp) // 64) * 64
        self.total = total

    def views(self, flat):
        return [flat[o:o + math.prod(s)].reshape(s) for o, s in zip(self.offs, self.shapes)]

    def fill(self, padded):
        """The buffer with every box cut from whole-domain arrays with ng
        ghost layers, one for each direction in ``dirs``."""
        flat = torch.zeros(self.total, dtype=torch.float64, device="cuda")
        q = 0
        vs = self.views(flat)
        for lo, _ in self.boxes:
            for a in padded:
                s = self.shapes[q]
                vs[q].copy_(a[lo[2]:lo[2] + s[0], lo[1]:lo[1] + s[1], lo[0]:lo[0] + s[2]])
                q += 1
        return flat.cpu().numpy() if self.host else flat


def _pad(a, bc, d, rule):
    """One ghost layer around a whole-domain array (d: face direction, -1
    cells): periodic images, else rule(direction, side) "edge" or "zero"."""
    for e in range(len(bc)):
        ax = 2 - e
        n = a.shape[ax]
        if bc[e][0] == PER:
            k = 1 if e == d else 0   # face n is face 0
            lo, hi = a.narrow(ax, n - 1 - k, 1), a.narrow(ax, k, 1)
        else:
            lo, hi = a.narrow(ax, 0, 1), a.narrow(ax, n - 1, 1)
            lo = lo if rule(e, 0) == "edge" else torch.zeros_like(lo)
            hi = hi if rule(e, 1) == "edge" else torch.zeros_like(hi)
        a = torch.cat([lo, a, hi], ax)
    return a


# ------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rand(g, *shape):
    return torch.rand(shape, dtype=torch.float64, device="cuda", generator=g)


def _randn(g, *shape):
    return torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)


def _face_shape(n, d):
    return tuple(n[e] + (e == d) for e in (2, 1, 0))


def _velocity(g, n, bc, scale=None):
    """U ~ U[-1, 1] on faces: one value per physical face, none through walls."""
    u = []
    for d in range(len(bc)):
        f = 2.0 * _rand(g, *_face_shape(n, d)) - 1.0
        if scale is not None:
            f = f * scale[d]
        ax = 2 - d
        if bc[d][0] == PER:
            f.narrow(ax, n[d], 1).copy_(f.narrow(ax, 0, 1))
        else:
            for s, at in ((0, 0), (1, n[d])):
                if bc[d][s] != OUT:
                    f.narrow(ax, at, 1).zero_()
        u.append(f)
    return u


def _planar(n, dim):
    """beta0 = exp(-r / H) of contrast 1e4 over the last direction: cells, edges."""
    nr = n[dim - 1]
    r = (torch.arange(nr, dtype=torch.float64, device="cuda") + 0.5) / nr
    e = torch.arange(nr + 1, dtype=torch.float64, device="cuda") / nr
    c = math.log(1e4)
    return torch.exp(-c * r), torch.exp(-c * e)


def _along(v, dim):
    return v.reshape((-1, 1, 1) if dim == 3 else (1, -1, 1))


def _means(a, d):
    """Mean of the two cells on every face of direction d (the end cells' own value on the domain's sides)."""
    ax = 2 - d
    p = torch.cat([a.narrow(ax, 0, 1), a, a.narrow(ax, a.shape[ax] - 1, 1)], ax)
    m = p.shape[ax] - 1
    return 0.5 * (p.narrow(ax, 0, m) + p.narrow(ax, 1, m))


def _star(n):
    """beta0 of a star on the cells: 1 at the centre to 1e-6 outside 0.45 of the shortest side."""
    h = 1.0 / max(n)
    c = [(torch.arange(n[d], dtype=torch.float64, device="cuda") + 0.5 - 0.5 * n[d]) * h for d in range(3)]
    r = torch.sqrt(c[2][:, None, None] ** 2 + c[1][None, :, None] ** 2 + c[0][None, None, :] ** 2)
    t = (1.0 - (r / (0.45 * min(n) * h)) ** 2).clamp_min(0.0)
    return (t ** 1.5).clamp_min(1e-6)


def _project_inputs(case, seed):
    """Whole-domain inputs of a projection: n, dim, bc, U, beta0 on faces (for
    the exact answer), rho with a ghost layer, macrhs, and the caller's beta0."""
    g, n, bc = _gen(seed), _ext(case), _bc(case)
    dim = len(bc)
    x = {"n": n, "dim": dim, "bc": bc, "h": 1.0 / max(n), "cart": None, "b0": None, "b0e": None, "macrhs": None}
    if case["beta0"] == "star":
        b = _star(n)
        rho = b * (1.0 + 0.005 * _randn(g, n[2], n[1], n[0]))
        x["cart"] = [_means(b, d) for d in range(3)]
        del b
        x["U"] = _velocity(g, n, bc, [_means(rho, d) ** -0.5 for d in range(3)])
    else:
        x["b0"], x["b0e"] = _planar(n, dim)
        rho = _along(x["b0"], dim) * (1.0 + 0.01 * _randn(g, n[2], n[1], n[0]))
        x["U"] = _velocity(g, n, bc)
        if case["macrhs"]:   # beta0 (S - Sbar): a heating-like source, smaller than div U
            x["macrhs"] = _along(x["b0"], dim) * _randn(g, n[2], n[1], n[0])
    x["rho"] = _pad(rho, bc, -1, lambda e, s: "edge")
    return x


def _umac_rule(bc, d):
    """What a face array of direction d holds beyond a physical side after a
    projection: an outlet copies its last face; a wall sets the tangential
    ghost to zero and leaves the normal one as it came in (zero here)."""
    return lambda e, s: "edge" if bc[e][s] == OUT else "zero"


def _layout(n, bc, boxes, h, **ng):
    dim = len(bc)
    return mac.Layout(dim=dim, boxes=boxes, domain_lo=(0,) * dim, domain_hi=tuple(n[d] - 1 for d in range(dim)),
                      dx=(h,) * dim, phys_bc=bc, **ng)


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"project": _prepare_project, "twolevel": _prepare_twolevel, "diffuse": _prepare_diffuse,
            "gradient": _prepare_gradient, "inputs": _prepare_inputs}[case["kind"]](case, seed)


def _table(arena, flat):
    return mac.PtrTable(arena.views(flat))


def _prepare_project(case, seed):
    x = _project_inputs(case, seed)
    n, dim, bc, host = x["n"], x["dim"], x["bc"], case["host"]
    boxes = _boxes(n, case["box"])
    au, ap = Arena(boxes, dim, list(range(dim)), 1, host), Arena(boxes, dim, [-1], 1, host)
    am = Arena(boxes, dim, [-1], 0, host)
    s = {"case": case, "u0": au.fill([_pad(x["U"][d], bc, d, lambda e, s: "zero") for d in range(dim)])}
    rho = ap.fill([x["rho"]])
    back = (lambda a: None if a is None else a.cpu().numpy()) if host else (lambda a: a)
    s["umac"] = s["u0"].copy() if host else s["u0"].clone()
    s["phi"] = np.zeros_like(rho) if host else torch.zeros_like(rho)
    cart = Arena(boxes, dim, list(range(dim)), 1)
    s["args"] = [_table(au, s["umac"]), _table(ap, s["phi"]), _table(ap, rho),
                 None if x["macrhs"] is None else _table(am, am.fill([x["macrhs"]])), back(x["b0"]), back(x["b0e"]),
                 None if x["cart"] is None else
                 _table(cart, cart.fill([_pad(x["cart"][d], bc, d, lambda e, s: "edge") for d in range(dim)]))]
    s["plan"] = mac.MacPlan(_layout(n, bc, boxes, x["h"]), mac.default_opts(
        precision=PREC[case["precision"]], omega=case["omega"], device_ptrs=int(not host)))
    return s


def _prepare_twolevel(case, seed):
    g, n = _gen(seed), _ext(case)
    bc = [[PER, PER], [PER, PER], [WALL, WALL]]
    r, m = (case["rx"], case["ry"], case["rz"]), (case["mx"], case["my"], case["mz"])
    s = {"case": case, "u0": [], "umac": [], "phi": [], "args": [[], [], [], [], []]}
    lays = []
    for l in range(2):
        f = l + 1
        org = tuple(2 * v for v in r) if l else (0, 0, 0)
        ext = tuple(2 * v for v in m) if l else n
        h = 1.0 / (max(n) * f)
        b0, b0e = _planar([f * v for v in n], 3)
        if l == 0:
            U = [_pad(u, bc, d, lambda e, s: "zero") for d, u in enumerate(_velocity(g, n, bc))]
            rho = _pad(_along(b0, 3) * (1.0 + 0.01 * _randn(g, n[2], n[1], n[0])), bc, -1, lambda e, s: "edge")
        else:   # the region with a ghost layer; below it the wall where it rests on the bottom
            U = [2.0 * _rand(g, *(v + 2 for v in _face_shape(ext, d))) - 1.0 for d in range(3)]
            if org[2] == 0:
                U[2][:2].zero_()
                for d in range(2):
                    U[d][:1].zero_()
            z = (torch.arange(org[2] - 1, org[2] + ext[2] + 1, device="cuda")).clamp(0, f * n[2] - 1)
            rho = _along(b0[z], 3) * (1.0 + 0.01 * _randn(g, ext[2] + 2, ext[1] + 2, ext[0] + 2))
        rel = _boxes(ext, case["box"])
        boxes = [tuple(tuple(v[e] + org[e] for e in range(3)) for v in b) for b in rel]
        au, ap = Arena(rel, 3, [0, 1, 2], 1), Arena(rel, 3, [-1], 1)
        u0, rf = au.fill(U), ap.fill([rho])
        s["u0"].append(u0)
        s["umac"].append(u0.clone())
        s["phi"].append(torch.zeros_like(rf))
        for q, a in enumerate((_table(au, s["umac"][l]), _table(ap, s["phi"][l]), _table(ap, rf), b0, b0e)):
            s["args"][q].append(a)
        lays.append(_layout([f * v for v in n], bc, boxes, h))
    s["plan"] = mac.MacMLPlan(lays, mac.default_opts(eps_rel=1e-9, precision=PREC[case["precision"]]))
    return s


def _diffuse_inputs(case, seed):
    """(alpha - D beta G) phi = rh of a thermal diffusion step: alpha the
    density, beta (dt / 2) k / c_p on faces with a diffusion number of about
    20 cells at the bottom, Dirichlet below (a ghost value), Neumann above."""
    g, n = _gen(seed), _ext(case)
    bc = [[PER, PER], [PER, PER], [mac.INLET, WALL]]
    h = 1.0 / max(n)
    b0, b0e = _planar(n, 3)
    alpha = _along(b0, 3) * (1.0 + 0.01 * _randn(g, n[2], n[1], n[0]))
    beta = []
    for d in range(3):
        f = 20.0 * h * h * (0.75 + 0.5 * _rand(g, *_face_shape(n, d))) * _along(b0e if d == 2 else b0, 3)
        if d < 2:
            f.narrow(2 - d, n[d], 1).copy_(f.narrow(2 - d, 0, 1))
        beta.append(f)
    old = 1.0 + 0.1 * _randn(g, n[2], n[1], n[0])
    low = 1.0 + 0.1 * _randn(g, 1, n[1], n[0])   # the boundary value on the bottom face
    rh = alpha * old
    return {"n": n, "bc": bc, "h": h, "alpha": alpha, "beta": beta, "old": old, "low": low, "rh": rh}


def _prepare_diffuse(case, seed):
    x = _diffuse_inputs(case, seed)
    n, bc = x["n"], x["bc"]
    boxes = _boxes(n, case["box"])
    a0, a1, af = Arena(boxes, 3, [-1], 0), Arena(boxes, 3, [-1], 1), Arena(boxes, 3, [0, 1, 2], 0)
    p = _pad(x["old"], bc, -1, lambda e, s: "zero")
    p[:1] = _pad(x["low"], bc[:2], -1, None)
    phi0 = a1.fill([p])
    fb = af.views(af.fill(x["beta"]))
    s = {"case": case, "phi0": phi0, "phi": phi0.clone(), "rh": a0.views(a0.fill([x["rh"]])),
         "alpha": a0.views(a0.fill([x["alpha"]])), "beta": [fb[3 * b:3 * b + 3] for b in range(len(boxes))]}
    s["boxes"] = a1.views(s["phi"])
    s["ell"] = [[mac.ELL_PER] * 2, [mac.ELL_PER] * 2, [mac.ELL_DIR, mac.ELL_NEU]]
    s["plan"] = mac.MacPlan(_layout(n, bc, boxes, x["h"]),
                            mac.default_opts(precision=PREC[case["precision"]], device_ptrs=1))
    return s


def _gradient_inputs(case, seed):
    """beta0 U, face coefficients beta0^2 / rho and the loss weights of a differentiable projection."""
    g, n = _gen(seed), _ext(case)
    bc = [[PER, PER], [PER, PER], [WALL, WALL]]
    b0, b0e = _planar(n, 3)
    rho = _pad(_along(b0, 3) * (1.0 + 0.01 * _randn(g, n[2], n[1], n[0])), bc, -1, lambda e, s: "edge")
    U = [u * _along(b0e if d == 2 else b0, 3) for d, u in enumerate(_velocity(g, n, bc))]
    sides = [(rho[1:-1, 1:-1, :-1], rho[1:-1, 1:-1, 1:]), (rho[1:-1, :-1, 1:-1], rho[1:-1, 1:, 1:-1]),
             (rho[:-1, 1:-1, 1:-1], rho[1:, 1:-1, 1:-1])]
    B = [(2.0 / (a + b) * _along(b0e if d == 2 else b0, 3) ** 2).contiguous() for d, (a, b) in enumerate(sides)]
    return {"n": n, "bc": bc, "h": 1.0 / max(n), "U": U, "B": B, "w": _randn(g, n[2], n[1], n[0])}


def _prepare_gradient(case, seed):
    x = _gradient_inputs(case, seed)
    return {"case": case, "U": [u.requires_grad_(True) for u in x["U"]], "B": [b.requires_grad_(True) for b in x["B"]],
            "w": x["w"], "plan": autograd.level_plan(x["n"], (x["h"],) * 3, x["bc"], precision=PREC[case["precision"]])}


def _sphere_inputs(case, seed):
    g, n = _gen(seed), _ext(case)
    h = 1.0 / max(n)
    dr = h / 5.0
    nr = int(0.5 * math.sqrt(sum(v * v for v in n)) * h / dr) + 2
    r = (torch.arange(nr, dtype=torch.float64, device="cuda") + 0.5) * dr
    rho0 = torch.exp(-8.0 * r * r)
    cells = lambda a: a * _randn(g, n[2], n[1], n[0])  # noqa: E731
    return {"n": n, "h": h, "dr": dr, "nr": nr, "beta0": rho0 ** 0.9, "Sbar": 0.1 * torch.cos(3.0 * r),
            "gamma1bar": 1.5 + 0.1 * r, "p0": rho0 ** 1.5 + 1e-4, "rho0": rho0, "S": cells(1.0), "dg": cells(0.01),
            "dp": cells(1e-3), "dchi": cells(1e-3), "dt": 0.01, "dpdt": 0.5, "cutoff": 0.1}


def _prepare_inputs(case, seed):
    x = _sphere_inputs(case, seed)
    n = x["n"]
    boxes = _boxes(n, case["box"])
    a0, af = Arena(boxes, 3, [-1], 0), Arena(boxes, 3, [0, 1, 2], 1)
    s = {"case": case, "x": {k: x[k] for k in ("beta0", "Sbar", "gamma1bar", "p0", "rho0", "dt", "dpdt", "cutoff")}}
    for k in ("S", "dg", "dp"):
        s[k] = a0.views(a0.fill([x[k]]))
    s["dchi0"] = a0.fill([x["dchi"]])
    s["dchi"], s["macrhs"] = s["dchi0"].clone(), torch.zeros_like(s["dchi0"])
    s["s0mac"] = torch.zeros(af.total, dtype=torch.float64, device="cuda")
    s["dchi_boxes"], s["macrhs_boxes"] = a0.views(s["dchi"]), a0.views(s["macrhs"])
    fb = af.views(s["s0mac"])
    s["s0mac_boxes"] = [fb[3 * b:3 * b + 3] for b in range(len(boxes))]
    s["sph"] = mac.sphr(x["dr"], x["nr"], [0.5 * v * x["h"] for v in n], (0.0, 0.0, 0.0), 3)
    s["plan"] = mac.MacPlan(_layout(n, [[OUT, OUT]] * 3, boxes, x["h"]), mac.default_opts(device_ptrs=1))
    return s


# -------------------------------------------------------------------- run
def run(s):
    case, plan = s["case"], s["plan"]
    kind = case["kind"]
    if kind == "project":
        if case["host"]:
            np.copyto(s["umac"], s["u0"])
            s["phi"].fill(0.0)
        else:
            s["umac"].copy_(s["u0"])
            s["phi"].zero_()
        plan.project(*s["args"])
        return {"umac": s["umac"], "phi": s["phi"]}
    if kind == "twolevel":
        for l in range(2):
            s["umac"][l].copy_(s["u0"][l])
            s["phi"][l].zero_()
        u, p, r, b0, b0e = s["args"]
        plan.project(u, p, r, None, b0, b0e)
        return {"umac": s["umac"], "phi": s["phi"]}
    if kind == "diffuse":
        s["phi"].copy_(s["phi0"])
        plan.solve(s["rh"], s["boxes"], s["beta"], s["alpha"], ell_bc=s["ell"], ng_phi=1)
        return {"phi": s["phi"]}
    if kind == "gradient":
        U, B = s["U"], s["B"]
        phi, *u = autograd.mac_project(plan, *U, *B)
        loss = (s["w"] * phi).sum() + 0.5 * sum((v * v).sum() for v in u)
        return {"phi": phi, "U": u, "grads": list(torch.autograd.grad(loss, U + B))}
    x = s["x"]
    s["dchi"].copy_(s["dchi0"])
    plan.make_macrhs(s["macrhs_boxes"], s["S"], s["dg"], x["Sbar"], x["beta0"], delta_p_term=s["dp"],
                     delta_chi=s["dchi_boxes"], gamma1bar=x["gamma1bar"], p0=x["p0"], rho0=x["rho0"], dt=x["dt"],
                     dpdt_factor=x["dpdt"], base_cutoff_density=x["cutoff"], is_predictor=False, sph=s["sph"])
    plan.make_s0mac(x["beta0"], s["sph"], s["s0mac_boxes"])
    return {"macrhs": s["macrhs"], "delta_chi": s["dchi"], "s0mac": s["s0mac"]}


def work(case):
    """Each input read once and each output written once; the arithmetic of
    the cycles that a rate of 0.08 a cycle needs (9 for ten digits, 8 sweeps'
    worth of 20 operations a cell on the finest level, an eighth or a quarter
    of a level below it)."""
    n = case["nx"] * case["ny"] * case["nz"]
    dim = 3 if case["nz"] > 1 else 2
    mg = 9 * 8 * 20 * (8.0 / 7.0 if dim == 3 else 4.0 / 3.0)
    kind = case["kind"]
    if kind == "project":
        b = 16 * dim + 16 + 8 + (8 if case["macrhs"] else 0) + (8 * dim if case["beta0"] == "star" else 0)
        return {"bytes": float(b * n), "flops": mg * n}
    if kind == "twolevel":
        n += 8 * case["mx"] * case["my"] * case["mz"]
        return {"bytes": 72.0 * n, "flops": mg * n}
    if kind == "diffuse":
        return {"bytes": 56.0 * n, "flops": mg * n}
    if kind == "gradient":   # U, beta, w in; phi, U and the gradients out
        return {"bytes": 8.0 * (6 + 1 + 4 + 6) * n, "flops": 2 * mg * n}
    return {"bytes": 8.0 * (4 + 2 + 3) * n, "flops": 100.0 * n}


# ------------------------------------------------------ exact answers, plain
def _fold(b, bc, d):
    """Face weights with the boundary conditions in them: Neumann 0, Dirichlet (value 0 on the face) twice beta."""
    b = b.clone()
    ax = 2 - d
    for s, at in ((0, 0), (1, b.shape[ax] - 1)):
        k = bc[s]
        if k != PER:
            b.narrow(ax, at, 1).mul_(2.0 if k == OUT else 0.0)
    return b


def _grad(p, d, per):
    """Differences of a cell array across every face of direction d (the
    periodic image, or 0, outside)."""
    ax = 2 - d
    n = p.shape[ax]
    lo, hi = (p.narrow(ax, n - 1, 1), p.narrow(ax, 0, 1)) if per else (torch.zeros_like(p.narrow(ax, 0, 1)),) * 2
    return torch.diff(torch.cat([lo, p, hi], ax), dim=ax)


class _Level:
    def __init__(self, w, ih2, per, alpha):
        self.w, self.ih2, self.per, self.alpha = w, ih2, per, alpha
        ref = w[0]
        self.shape = (ref.shape[0], ref.shape[1], ref.shape[2] - 1)
        diag = torch.zeros(self.shape, dtype=torch.float64, device="cuda") if alpha is None else alpha.clone()
        for d in range(len(w)):
            ax = 2 - d
            m = self.shape[ax]
            diag += ih2[d] * (w[d].narrow(ax, 0, m) + w[d].narrow(ax, 1, m))
        self.idiag = 1.0 / diag

    def apply(self, p):
        out = torch.zeros_like(p) if self.alpha is None else self.alpha * p
        for d in range(len(self.w)):
            out -= self.ih2[d] * torch.diff(self.w[d] * _grad(p, d, self.per[d]), dim=2 - d)
        return out

    def coarser(self):
        dim = len(self.w)
        if any(self.shape[2 - d] % 2 or self.shape[2 - d] < 4 for d in range(dim)):
            return None

        def pairs(a, ax):
            return 0.5 * (a[(slice(None),) * ax + (slice(0, None, 2),)] + a[(slice(None),) * ax + (slice(1, None, 2),)])

        w = []
        for d in range(dim):
            a = self.w[d][(slice(None),) * (2 - d) + (slice(0, None, 2),)]
            for e in range(dim):
                if e != d:
                    a = pairs(a, 2 - e)
            w.append(a)
        alpha = self.alpha
        if alpha is not None:
            for e in range(dim):
                alpha = pairs(alpha, 2 - e)
        return _Level(w, [v / 4.0 for v in self.ih2], self.per, alpha)


def _mg_solve(w, ih2, per, rhs, singular, alpha=None, tol=1e-14):
    """Conjugate gradients with a multigrid preconditioner, to rounding."""
    levels = [_Level(w, ih2, per, alpha)]
    while True:
        c = levels[-1].coarser()
        if c is None:
            break
        levels.append(c)
    L = levels[-1]
    m = math.prod(L.shape)
    eye = torch.eye(m, dtype=torch.float64, device="cuda")
    A = torch.stack([L.apply(eye[q].reshape(L.shape)).reshape(-1) for q in range(m)])
    if singular:
        A += float(A.diagonal().mean()) / m
    bottom = torch.linalg.inv(A)
    three = len(w) == 3

    def cycle(l, r):
        L = levels[l]
        if l == len(levels) - 1:
            return (bottom @ r.reshape(-1)).reshape(r.shape)
        x = 0.8 * L.idiag * r
        x += 0.8 * L.idiag * (r - L.apply(x))
        d = (r - L.apply(x))[None, None]
        d = torch.nn.functional.avg_pool3d(d, 2) if three else torch.nn.functional.avg_pool2d(d[0], 2)[None]
        e = cycle(l + 1, d[0, 0])
        if three:
            x += torch.nn.functional.interpolate(e[None, None], scale_factor=2, mode="trilinear")[0, 0]
        else:
            x += torch.nn.functional.interpolate(e[None], scale_factor=2, mode="bilinear")[0]
        for _ in range(2):
            x += 0.8 * L.idiag * (r - L.apply(x))
        return x

    if singular:
        rhs = rhs - rhs.mean()
    x, r = torch.zeros_like(rhs), rhs.clone()
    norm = float(rhs.norm())
    z = cycle(0, r)
    p, rz = z.clone(), float((r * z).sum())
    best, since = norm, 0
    for _ in range(100):
        Ap = levels[0].apply(p)
        a = rz / float((p * Ap).sum())
        x += a * p
        rn = r - a * Ap
        now = float(rn.norm())
        if now <= tol * norm:
            break
        best, since = (now, 0) if now < 0.9 * best else (best, since + 1)
        if since >= 4:   # at rounding
            break
        z = cycle(0, rn)
        b = float((z * (rn - r)).sum()) / rz
        r, rz = rn, float((rn * z).sum())
        p = z + b * p
    return x - x.mean() if singular else x


def exact(case, seed):
    """What ``run`` returns, from plain torch in 64 bits.  Where the problem
    is singular the library's phi is defined up to a constant, so it has no
    such value; the composite operator of two levels is solved nowhere else in
    seconds."""
    kind = case["kind"]
    if kind == "project":
        return _exact_project(case, seed)
    if kind == "diffuse":
        return _exact_diffuse(case, seed)
    if kind == "gradient":
        return _exact_gradient(case, seed)
    if kind == "inputs":
        return _exact_inputs(case, seed)
    return None


def _exact_project(case, seed):
    x = _project_inputs(case, seed)
    n, dim, bc, h = x["n"], x["dim"], x["bc"], x["h"]
    per = [bc[d][0] == PER for d in range(dim)]
    singular = all(k != OUT for b in bc for k in b)
    b0f, w = [], []
    for d in range(dim):
        b0f.append(x["cart"][d] if x["cart"] is not None else _along(x["b0e"] if d == dim - 1 else x["b0"], dim))
        ax = 2 - d
        r = x["rho"]
        for e in range(dim):
            if e != d:
                r = r.narrow(2 - e, 1, n[e])
        w.append(_fold(2.0 / (r.narrow(ax, 0, n[d] + 1) + r.narrow(ax, 1, n[d] + 1)) * b0f[d] ** 2, bc[d], d))
    div = sum(torch.diff(x["U"][d] * b0f[d], dim=2 - d) / h for d in range(dim))
    rhs = -div if x["macrhs"] is None else x["macrhs"] - div
    phi = _mg_solve(w, [1.0 / h ** 2] * dim, per, rhs, singular)
    U = [x["U"][d] - w[d] * _grad(phi, d, per[d]) / h / b0f[d] for d in range(dim)]
    boxes = _boxes(n, case["box"])
    au, ap = Arena(boxes, dim, list(range(dim)), 1, case["host"]), Arena(boxes, dim, [-1], 1, case["host"])
    out = {"umac": au.fill([_pad(U[d], bc, d, _umac_rule(bc, d)) for d in range(dim)]), "phi": None}
    if not singular:
        walls = [[WALL, WALL]] * dim   # phi's ghost cells stay as they came in, zero
        flat = ap.fill([_pad(phi, walls, -1, lambda e, s: "zero")])
        for (lo, hi), v in zip(boxes, ap.views(flat)):   # between boxes too
            for e in range(dim):
                for at in (0, hi[e] - lo[e] + 2):
                    v[(slice(None),) * (2 - e) + (at,)] = 0.0
        out["phi"] = flat
    return out


def _exact_diffuse(case, seed):
    x = _diffuse_inputs(case, seed)
    n, h = x["n"], x["h"]
    w = [b.clone() for b in x["beta"]]
    w[2][:1] *= 2.0
    w[2][-1:] = 0.0
    rhs = x["rh"].clone()
    rhs[:1] += w[2][:1] * x["low"] / h ** 2
    phi = _mg_solve(w, [1.0 / h ** 2] * 3, [True, True, False], rhs, False, alpha=x["alpha"])
    boxes = _boxes(n, case["box"])
    a1 = Arena(boxes, 3, [-1], 1)
    bc = x["bc"]
    p = _pad(x["old"], bc, -1, lambda e, s: "zero")
    p[:1] = _pad(x["low"], bc[:2], -1, None)
    flat = a1.fill([p])
    for (lo, hi), v in zip(boxes, a1.views(flat)):   # the solution on the valid cells, the ghosts untouched
        v[1:-1, 1:-1, 1:-1] = phi[lo[2]:hi[2] + 1, lo[1]:hi[1] + 1, lo[0]:hi[0] + 1]
    return {"phi": flat}


def _exact_gradient(case, seed):
    x = _gradient_inputs(case, seed)
    n, h, bc = x["n"], x["h"], x["bc"]
    per = [True, True, False]
    w = [_fold(x["B"][d], bc[d], d) for d in range(3)]
    ih2 = [1.0 / h ** 2] * 3
    phi = _mg_solve(w, ih2, per, -sum(torch.diff(x["U"][d], dim=2 - d) / h for d in range(3)), True)
    G = [_grad(phi, d, per[d]) / h for d in range(3)]
    U = [x["U"][d] - w[d] * G[d] for d in range(3)]
    # the adjoint: A lambda = dL/dphi - G^T (w dL/dU) with dL/dU = U
    p = torch.zeros_like(phi).requires_grad_(True)
    gt = torch.autograd.grad(sum((U[d] * w[d] * _grad(p, d, per[d]) / h).sum() for d in range(3)), p)[0]
    lam = _mg_solve(w, ih2, per, x["w"] - gt, True)
    gU, gB = [], []
    for d in range(3):
        dt = -_grad(lam, d, False) / h   # D^T lambda over the cells that exist
        gU.append(U[d] - dt)
        b = G[d] * (dt - U[d])
        if not per[d]:   # no flux through the walls
            b[:1] = 0.0
            b[-1:] = 0.0
        gB.append(b)
    return {"phi": phi, "U": U, "grads": gU + gB}


def _radial(s0, x):
    """The quadratic radial interpolation of a profile on the cells, limited to its three points' range."""
    n, h, dr, nr = x["n"], x["h"], x["dr"], x["nr"]
    c = [(torch.arange(n[d], dtype=torch.float64, device="cuda") + 0.5) * h - 0.5 * n[d] * h for d in range(3)]
    r = torch.sqrt(c[0][None, None, :] ** 2 + c[1][None, :, None] ** 2 + c[2][:, None, None] ** 2)
    q = (r / dr).long().clamp(1, nr - 2)
    xs = [(q + o + 0.5) * dr for o in (-1, 0, 1)]
    y = [s0[q + o] for o in (-1, 0, 1)]
    s01, s12 = (y[1] - y[0]) / (xs[1] - xs[0]), (y[2] - y[1]) / (xs[2] - xs[1])
    v = y[0] + s01 * (r - xs[0]) + (s12 - s01) / (xs[2] - xs[0]) * (r - xs[0]) * (r - xs[1])
    lo, hi = torch.minimum(torch.minimum(y[0], y[1]), y[2]), torch.maximum(torch.maximum(y[0], y[1]), y[2])
    return torch.minimum(torch.maximum(v, lo), hi)


def _exact_inputs(case, seed):
    x = _sphere_inputs(case, seed)
    n = x["n"]
    b0, sb, g1, p0, r0 = (_radial(x[k], x) for k in ("beta0", "Sbar", "gamma1bar", "p0", "rho0"))
    on = r0 > x["cutoff"]
    dchi = torch.where(on, x["dchi"] + x["dpdt"] * x["dp"] / (x["dt"] * g1 * p0), x["dchi"])
    rhs = b0 * (x["S"] - sb + x["dg"]) + torch.where(on, b0 * dchi, torch.zeros_like(dchi))
    boxes = _boxes(n, case["box"])
    a0, af = Arena(boxes, 3, [-1], 0), Arena(boxes, 3, [0, 1, 2], 1)
    open_ = [[OUT, OUT]] * 3
    edge = lambda e, s: "edge"  # noqa: E731
    c = _pad(_pad(b0, open_, -1, edge), open_, -1, edge)   # two layers: the faces of the grown boxes
    m = [0.5 * (c.narrow(2 - d, 0, n[d] + 3) + c.narrow(2 - d, 1, n[d] + 3)) for d in range(3)]
    for d in range(3):
        for e in range(3):
            if e != d:
                m[d] = m[d].narrow(2 - e, 1, n[e] + 2)
    return {"macrhs": a0.fill([rhs]), "delta_chi": a0.fill([dchi]), "s0mac": af.fill(m)}
