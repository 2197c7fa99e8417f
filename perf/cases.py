"""What the speed of this framework is measured on: pressure solves as a fluid
simulation asks for them, through the public entry points (`uaamg_amd.Context`,
`Batch`, `Server`, `Lib.amgpcg`).

A case is one of six kinds of work:
  frame    one time step's solve with host arrays and a mask that is sent again
           (what the C++ solver plugin does on every call)
  solve    one solve on device arrays; `moving`: the solids moved, so the
           hierarchy is rebuilt from the mask; `warm`: it starts from the
           previous step's pressure
  project  the MAC velocity projection around the solve, on device arrays
  batch    many independent grids in one call
  serve    one frame of each of many simulations through the request loop
  amgpcg   the standalone Ax = b entry point (host arrays)

Grids are the reference layout: padded arrays, x fastest, h = L/n.  The
divergence of a smooth random velocity field (a lattice of normals, upsampled,
plus 2 % grid noise; zero on walls and solid faces) is the right-hand side;
solids are disjoint balls, with a floor slab in the plume.  A form that
computes in FP32 hands its pressure on in FP32, as an FP32 simulation keeps
it; FP64 forms return FP64.
"""
import ctypes
import math
import random

import numpy as np
import torch
import torch.nn.functional as F

import uaamg_amd as U
from uaamg_amd import capi

PRECISION = {"fp64": U.FP64, "fp32": U.FP32, "bf16": U.MIXED_BF16, "bf16r": U.MIXED_BF16R, "mixed64": U.MIXED_F64}
PRECOND = {"uaamg": U.PRECOND_UAAMG, "gmg": U.PRECOND_GMG, "amg": U.PRECOND_AMG}
HIERARCHY = {"reference": U.HIERARCHY_REFERENCE, "keep_fluid": U.HIERARCHY_KEEP_FLUID}
#: boundary types: all walls closed, or the +x face an outlet (p = 0)
WALLS = {"closed": [0, 0, 0, 0, 0, 0], "outlet": [0, 1, 0, 0, 0, 0]}
DT = 1e-2
MAX_ITER = 2000


def _solve(name, nx, ny, nz, **kw):
    c = {"name": name, "kind": "solve", "nx": nx, "ny": ny, "nz": nz, "precision": "fp32", "precond": "uaamg",
         "hierarchy": "reference", "walls": "closed", "balls": 3, "slab": False, "stretch": 1.0, "moving": True,
         "warm": False, "tol": 1e-6}
    c.update(kw)
    return c


def listed():
    return [
        # an interactive 2D simulation through the solver plugin: the mask and
        # the arrays come from the host at every frame (the reference's default
        # FP64 form, a test-sized grid); latency and launches count
        _solve("frame2d_64x48", 64, 48, 1, kind="frame", precision="fp64", balls=1),
        # a small 3D simulation on the device, static solids, warm start, the
        # hierarchy with the fewest iterations: a real-time user's choice
        _solve("warm3d_48x40x36", 48, 40, 36, hierarchy="keep_fluid", balls=2, moving=False, warm=True, tol=1e-5),
        # the 1024 x 512 MAC grid with a disc and dx != dy, FP64 as the
        # reference runs it
        _solve("mac2d_1024x512", 1024, 512, 1, precision="fp64", balls=1, stretch=512 / 480),
        # the reference's default 2D keys "pcg" / "pcg_gmg", sides that are not
        # powers of two
        _solve("gmg2d_500x390", 500, 390, 1, precision="fp64", precond="gmg", balls=2),
        # the buoyant-plume scene at 256^3 (the headline benchmark's size and
        # form): solids moved, cold start
        _solve("plume3d_256", 256, 256, 256, balls=8, slab=True),
        # the 256 x 128 x 128 channel that the reference's published figures
        # are quoted on: FP64, no solids, one grid for the whole run
        _solve("channel3d_256x128_fp64", 256, 128, 128, precision="fp64", balls=0, moving=False),
        # odd, ragged sides, an outlet, several solids
        _solve("ragged3d_151x97x63", 151, 97, 63, walls="outlet", balls=3),
        # a long wind tunnel with obstacles, the largest grid here: rows wider
        # than 256 cells
        _solve("tunnel3d_512x256x256", 512, 256, 256, walls="outlet", balls=4, moving=False),
        # the pressure step of a projection method with moving solids, FP64
        _solve("project3d_128x64x64", 128, 64, 64, kind="project", precision="fp64", balls=2),
        # an ensemble of independent 2D and 3D grids of uneven size
        {"name": "batch_18", "kind": "batch", "precision": "fp32", "n2d": 12, "n3d": 6, "lo2d": 64, "hi2d": 768,
         "lo3d": 32, "hi3d": 128, "hierarchy": "reference", "tol": 1e-6},
        # one frame of each of 16 served simulations, warm start, BF16 levels
        {"name": "serve_16", "kind": "serve", "precision": "bf16", "n2d": 8, "n3d": 8, "lo2d": 64, "hi2d": 768,
         "lo3d": 32, "hi3d": 128, "hierarchy": "reference", "tol": 1e-5},
        # the standalone dense-grid entry point, host arrays
        {"name": "amgpcg_256", "kind": "amgpcg", "n": 256, "precision": "fp64", "tol": 1e-8},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, dim, lo, hi, most):
    """Sides between lo and hi with at most `most` cells, aspect ratios up to 3."""
    cells = math.exp(rng.uniform(math.log(lo ** dim), math.log(most)))
    w = [math.exp(rng.uniform(-0.55, 0.55)) for _ in range(dim)]
    s = (cells / math.prod(w)) ** (1.0 / dim)
    n = [min(hi, max(lo, int(round(s * v)))) for v in w]
    while math.prod(n) > most:
        k = n.index(max(n))
        n[k] = int(n[k] * 0.95)
    return n + [1] * (3 - dim)


def draw(rng):
    kind = rng.choice(["solve3d"] * 6 + ["solve2d"] * 3 + ["frame", "project", "batch", "serve", "amgpcg"])
    if kind in ("batch", "serve"):
        lo2, lo3 = _logint(rng, 48, 96), _logint(rng, 24, 40)
        return {"kind": kind, "precision": rng.choice(["fp32", "bf16"]), "n2d": rng.randint(4, 10), "n3d": rng.randint(2, 5),
                "lo2d": lo2, "hi2d": lo2 * rng.randint(3, 7), "lo3d": lo3, "hi3d": lo3 * rng.randint(2, 3),
                "hierarchy": rng.choice(["reference", "keep_fluid"]), "tol": 1e-5 if kind == "serve" else 1e-6}
    if kind == "amgpcg":
        p = rng.choice(["fp64", "fp32"])
        return {"kind": kind, "n": _logint(rng, 31, 700), "precision": p, "tol": 1e-8 if p == "fp64" else 1e-5}
    kw = {"balls": rng.randint(0, 4), "walls": rng.choice(["closed", "closed", "outlet"]), "hierarchy": rng.choice(["reference", "reference", "keep_fluid"]),
          "stretch": rng.choice([1.0, 1.0, round(rng.uniform(0.8, 1.25), 3)])}
    if kind == "solve3d":
        p = rng.choice(["fp32", "fp32", "fp32", "bf16", "bf16r", "fp64", "fp64", "mixed64"])
        n = _sides(rng, 3, 16, 512, 256 ** 3 if p in ("fp32", "bf16r") else 160 ** 3)
        kw.update(precision=p, slab=rng.random() < 0.3, moving=rng.random() < 0.5, warm=rng.random() < 0.4)
        kw["tol"] = 1e-5 if kw["warm"] else 1e-6
    elif kind == "solve2d":
        p = rng.choice(["fp64", "fp64", "fp32", "mixed64"])
        n = _sides(rng, 2, 32, 2048, 1 << 20)
        kw.update(precision=p, precond=rng.choice(["uaamg", "uaamg", "gmg", "amg"]), moving=rng.random() < 0.5, warm=rng.random() < 0.4)
        kw["tol"] = 1e-5 if kw["warm"] else 1e-6
        if kw["precond"] != "uaamg":      # these two are the reference's, which has closed walls only
            kw.update(walls="closed", hierarchy="reference")
    elif kind == "frame":
        dim = rng.choice([2, 3])
        n = _sides(rng, dim, 16, 256, 128 ** 2 if dim == 2 else 48 ** 3)
        kw.update(kind=kind, precision=rng.choice(["fp64", "fp64", "fp32"]))
    else:
        dim = rng.choice([2, 3, 3])
        n = _sides(rng, dim, 16, 512, 400 ** 2 if dim == 2 else 112 ** 3)
        kw.update(kind=kind, precision=rng.choice(["fp64", "fp32"]))
    c = _solve("", *n, **kw)
    del c["name"]
    return c


# ---- inputs ----

def _dims(case):
    return (case["nx"], case["ny"]) if case["nz"] == 1 else (case["nx"], case["ny"], case["nz"])


def _spacing(n, stretch):
    """Cells of 1/max(n); `stretch` scales the y spacing."""
    return tuple((stretch if a == 1 else 1.0) / max(n) for a in range(len(n)))


def _solid(n, h, balls, slab, r, dev):
    """Padded mask [k][j][i]: disjoint balls clear of the walls and of each
    other by at least 2.5 cells, and a floor slab (so the fluid is connected)."""
    dim, ext = len(n), [n[a] * h[a] for a in range(len(n))]
    lmin, gap = min(ext), 2.5 * max(h)
    shape = tuple(v + 2 for v in reversed(n))
    solid = torch.zeros(shape, dtype=torch.bool, device=dev)
    x = [((torch.arange(n[a] + 2, device=dev, dtype=torch.float64) - 0.5) * h[a]).reshape([-1 if b == dim - 1 - a else 1 for b in range(dim)]) for a in range(dim)]
    floor = 0.1 * ext[1] if slab else 0.0
    if slab:
        solid |= x[1] < floor
    put = []
    for _ in range(balls):
        for _try in range(20):
            rad = r.uniform(0.06, 0.13) * lmin
            lo = [rad + gap + (floor if a == 1 else 0.0) for a in range(dim)]
            if any(lo[a] >= ext[a] - rad - gap for a in range(dim)):
                continue
            cen = [r.uniform(lo[a], ext[a] - rad - gap) for a in range(dim)]
            if all(math.dist(cen, c) > rad + q + gap for c, q in put):
                put.append((cen, rad))
                solid |= sum((x[a] - cen[a]) ** 2 for a in range(dim)) < rad * rad
                break
    return solid


def _smooth(size, gen, dev):
    """A lattice of normals upsampled to `size`, with 2 % grid noise."""
    lat = torch.randn([1, 1] + [min(12, max(2, s // 6)) for s in size], dtype=torch.float64, generator=gen).to(dev)
    f = F.interpolate(lat, size=list(size), mode="trilinear" if len(size) == 3 else "bilinear", align_corners=True)[0, 0]
    dgen = torch.Generator(device=dev)
    dgen.manual_seed(int(torch.randint(1 << 40, (1,), generator=gen)))
    return f + 0.02 * torch.randn(f.shape, dtype=torch.float64, device=dev, generator=dgen)


def _velocity(n, solid, gen, dev):
    """MAC face arrays [u, v(, w)]: zero on wall faces and on faces of solid cells."""
    dim, out = len(n), []
    for a in range(dim):
        ax = dim - 1 - a                                   # array axis of direction a
        size = [v for v in reversed(n)]
        size[ax] -= 1
        shape = [v + 2 for v in reversed(n)]
        shape[ax] -= 1
        f = torch.zeros(shape, dtype=torch.float64, device=dev)
        f[(slice(1, -1),) * dim] = _smooth(size, gen, dev)
        s = solid.narrow(ax, 0, n[a] + 1) | solid.narrow(ax, 1, n[a] + 1)
        f[s] = 0.0
        out.append(f)
    return out


def _div(n, h, vel, fluid):
    """Padded div(u)/dt on fluid cells."""
    dim = len(n)
    rhs = torch.zeros(fluid.shape, dtype=torch.float64, device=fluid.device)
    for a in range(dim):
        ax, f = dim - 1 - a, vel[a][tuple(slice(None) if b == dim - 1 - a else slice(1, -1) for b in range(dim))]
        rhs[(slice(1, -1),) * dim] += (f.narrow(ax, 1, n[a]) - f.narrow(ax, 0, n[a])) / (h[a] * DT)
    rhs[~fluid] = 0.0
    return rhs


def _fluid(solid):
    fl = torch.zeros_like(solid)
    inner = (slice(1, -1),) * solid.dim()
    fl[inner] = ~solid[inner]
    return fl


def _scene(n, stretch, balls, slab, walls, warm, seed, velocity=False, dev=None):
    """One frame's inputs, made from the seed alone."""
    dev = dev or torch.device("cuda")
    r = random.Random(seed)
    gen = torch.Generator()
    gen.manual_seed(seed)
    h = _spacing(n, stretch)
    solid = _solid(n, h, balls, slab, r, dev)
    fluid = _fluid(solid)
    vel = _velocity(n, solid, gen, dev)
    rhs = _div(n, h, vel, fluid)
    s = {"n": n, "h": h, "wall": WALLS[walls], "solid": solid.to(torch.uint8).reshape(-1).contiguous(), "fluid": fluid, "rhs": rhs}
    if warm:   # the previous step's pressure solves the previous step's equation; the new one differs by a tenth
        p0 = torch.zeros_like(rhs)
        p0[(slice(1, -1),) * len(n)] = _smooth([v for v in reversed(n)], gen, dev)
        p0[~fluid] = 0.0
        if not any(s["wall"]):
            p0[fluid] -= p0[fluid].mean()
        A = _Operator(n, h, fluid, s["wall"])
        old = -A(p0)
        s["rhs"] = old + rhs * (0.1 * float(old.norm() / rhs.norm().clamp_min(1e-30)))
        s["p0"] = p0
    if velocity:
        s["vel"] = vel
    return s


def _members(case, seed):
    """The grids of a batch or of a server: square / cubic, log-uniform sides, 0-3 balls."""
    r = random.Random(seed * 7919 + 1)
    out = []
    sizes = random.Random(17)      # the same mix of sizes for every seed: a user's set of simulations
    for k in range(case["n2d"] + case["n3d"]):
        dim, (lo, hi) = (2, (case["lo2d"], case["hi2d"])) if k < case["n2d"] else (3, (case["lo3d"], case["hi3d"]))
        n = (_logint(sizes, lo, hi),) * dim
        walls = "outlet" if sizes.random() < 0.25 else "closed"
        out.append(_scene(n, 1.0, r.randint(0, 3), False, walls, case["kind"] == "serve", r.randrange(1 << 40)))
    return out


def _amg_rhs(n, seed):
    r = np.random.default_rng(seed)
    b = np.zeros((n + 2, n + 2))
    t = np.arange(1, n + 1) / (n + 1)
    for _ in range(4):
        k, l = r.integers(1, 6, 2)
        b[1:-1, 1:-1] += r.uniform(-20, 20) * np.outer(np.sin(np.pi * k * t), np.sin(np.pi * l * t))
    b[1:-1, 1:-1] += 0.1 * r.standard_normal((n, n))
    return b.reshape(-1)


def _opts(case):
    return {"precision": PRECISION[case["precision"]], "tol_mode": U.TOL_REL, "max_iter": MAX_ITER, "tol": case["tol"],
            "hierarchy_mode": HIERARCHY[case["hierarchy"]]}


def _out(case, t):
    return t if case["precision"] in ("fp64", "mixed64") else t.float()


def _device_grid(s):
    g = capi.make_grid(s["n"], s["h"], np.zeros(1, np.uint8), s["wall"])
    g.solid = ctypes.c_void_p(s["solid"].data_ptr())
    return g


def _set_grid_device(ctx, s, grid):
    ctx.n, ctx.dim, ctx.N = s["n"], len(s["n"]), s["rhs"].numel()
    rc = ctx.lib.L.uaamg_set_grid_device(ctx.h, ctypes.byref(grid))
    if rc != U.OK:
        raise RuntimeError(f"set_grid_device: {U.status_name(rc)}")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "amgpcg":
        b = _amg_rhs(case["n"], seed)
        return {"case": case, "b": b, "tol": case["tol"] * float(np.linalg.norm(b)), "lib": U.load()}
    if kind in ("batch", "serve"):
        m = _members(case, seed)
        for s in m:
            s["p"] = torch.zeros_like(s["rhs"])
        torch.cuda.synchronize()
        if kind == "batch":
            b = U.Batch(use_graph=1, **_opts(case))
            for s in m:
                b.add(s["n"], s["h"], s["solid"].data_ptr(), s["wall"], device=True)
            return {"case": case, "members": m, "batch": b}
        srv = U.Server(8 << 30, max_active=64, use_graph=1, **_opts(case))
        for k, s in enumerate(m):
            srv.register(k, s["n"], s["h"], s["solid"].cpu().numpy(), s["wall"])
        return {"case": case, "members": m, "server": srv}
    s = _scene(_dims(case), case["stretch"], case["balls"], case["slab"], case["walls"], case["warm"], seed, kind == "project")
    ctx = U.Context(preconditioner=PRECOND[case["precond"]], **_opts(case))
    if kind == "frame":
        return {"case": case, "ctx": ctx, "n": s["n"], "h": s["h"], "wall": s["wall"], "solid": s["solid"].cpu().numpy(), "rhs": s["rhs"].reshape(-1).cpu().numpy()}
    s["p"] = torch.zeros_like(s["rhs"])
    s["grid"] = _device_grid(s)
    torch.cuda.synchronize()
    _set_grid_device(ctx, s, s["grid"])
    if kind == "project":
        s["face"] = [f.clone() for f in s["vel"]]
    s.update(case=case, ctx=ctx)
    torch.cuda.synchronize()
    return s


# ---- one pass ----

def _ready():
    """The library works on streams of its own: what torch's stream wrote has to be there."""
    torch.cuda.current_stream().synchronize()


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "frame":
        state["ctx"].set_grid(state["n"], state["h"], state["solid"], state["wall"])
        p, _ = state["ctx"].solve(state["rhs"], MAX_ITER, case["tol"])
        return p if case["precision"] == "fp64" else p.astype(np.float32)
    if kind == "amgpcg":
        x, _ = state["lib"].amgpcg(case["n"], state["b"], MAX_ITER, state["tol"], PRECISION[case["precision"]])
        return x if case["precision"] == "fp64" else x.astype(np.float32)
    if kind == "batch":
        m = state["members"]
        for s in m:
            s["p"].zero_()
        _ready()
        state["batch"].solve_device([s["rhs"].data_ptr() for s in m], [s["p"].data_ptr() for s in m], None, MAX_ITER, case["tol"])
        return [_out(case, s["p"]) for s in m]
    if kind == "serve":
        m, srv = state["members"], state["server"]
        for s in m:
            s["p"].copy_(s["p0"])
        _ready()
        for k, s in enumerate(m):
            srv.submit(k, s["rhs"].data_ptr(), s["p"].data_ptr(), 1, MAX_ITER, case["tol"])
        left = len(m)
        while left:
            left -= len(srv.step())
        return [_out(case, s["p"]) for s in m]
    ctx = state["ctx"]
    if case["moving"]:
        _set_grid_device(ctx, state, state["grid"])
    if kind == "project":
        for f, f0 in zip(state["face"], state["vel"]):
            f.copy_(f0)
        _ready()
        ptr = [f.data_ptr() for f in state["face"]] + [None]
        ctx.project_device(ptr[0], ptr[1], ptr[2], state["p"].data_ptr(), DT, MAX_ITER, case["tol"])
        return [_out(case, f) for f in state["face"]] + [_out(case, state["p"])]
    if case["warm"]:
        state["p"].copy_(state["p0"])
    else:
        state["p"].zero_()
    _ready()
    ctx.solve_device(state["rhs"].data_ptr(), state["p"].data_ptr(), int(case["warm"]), MAX_ITER, case["tol"])
    return _out(case, state["p"])


def work(case):
    """Mask, right-hand side (or velocities) and, on a warm start, the old
    pressure read once, the pressure (and velocities) written once; and for
    the operations one application of the 5- / 7-point operator: an iterative
    method repeats that, but how often depends on the method."""
    if case["kind"] == "amgpcg":
        return {"bytes": 16 * case["n"] ** 2, "flops": 6 * case["n"] ** 2}
    if case["kind"] in ("batch", "serve"):
        sizes, b, f = random.Random(17), 0, 0
        for k in range(case["n2d"] + case["n3d"]):
            two = k < case["n2d"]
            side = _logint(sizes, case["lo2d"] if two else case["lo3d"], case["hi2d"] if two else case["hi3d"])
            sizes.random()
            cells = side ** 2 if two else side ** 3
            b += cells * (17 if case["kind"] == "batch" else 25)
            f += cells * (9 if two else 13)
        return {"bytes": b, "flops": f}
    cells, dim = case["nx"] * case["ny"] * case["nz"], 2 if case["nz"] == 1 else 3
    bytes_ = cells * (1 + 16 * dim + 8) if case["kind"] == "project" else cells * (17 + 8 * case["warm"])
    return {"bytes": bytes_, "flops": cells * (4 * dim + 1)}


# ---- the same results in 64 bits, by plain torch ----

class _Operator:
    """A = -laplacian on the fluid cells, p = 0 on outlet walls (half a cell away)."""

    def __init__(self, n, h, fluid, wall):
        self.dim, self.n = len(n), n
        self.ih2 = [1.0 / (v * v) for v in h]
        self.inner = (slice(1, -1),) * self.dim
        f = fluid.to(torch.float64)
        self.face, self.diag = [], torch.zeros_like(f)
        for a in range(self.dim):
            ax = self.dim - 1 - a
            c = f.narrow(ax, 0, n[a] + 1) * f.narrow(ax, 1, n[a] + 1) * self.ih2[a]
            self.face.append(c)
            self.diag.narrow(ax, 0, n[a] + 1).add_(c)
            self.diag.narrow(ax, 1, n[a] + 1).add_(c)
        self.wall = torch.zeros_like(f)
        for k in range(2 * self.dim):
            if wall[k]:
                ax = self.dim - 1 - k // 2
                at = 1 if k % 2 == 0 else n[k // 2]
                self.wall.select(ax, at).add_(2.0 * self.ih2[k // 2])
        self.wall *= f
        self.diag += self.wall
        self.open = bool(self.wall.any())

    def __call__(self, p):
        out = self.wall * p
        for a in range(self.dim):
            ax = self.dim - 1 - a
            n = self.n[a] + 1
            flux = (p.narrow(ax, 1, n) - p.narrow(ax, 0, n)).mul_(self.face[a])
            out.narrow(ax, 0, n).sub_(flux)
            out.narrow(ax, 1, n).add_(flux)
        return out


def _pressure(n, h, fluid, wall, rhs, relres=1e-10):
    """lap(p) = rhs by Jacobi-preconditioned CG; zero mean where all walls are closed."""
    A = _Operator(n, h, fluid, wall)
    f = fluid.to(torch.float64)
    cells = f.sum()
    b = -rhs * f
    if not A.open:
        b -= f * (b.sum() / cells)
    w = torch.where(A.diag > 0, 1.0 / A.diag.clamp_min(1e-300), torch.zeros_like(A.diag))
    x, r = torch.zeros_like(b), b.clone()
    z = w * r
    d, rz, stop = z.clone(), (r * z).sum(), float(b.norm()) * relres
    for k in range(60000):
        q = A(d)
        alpha = rz / (d * q).sum()
        x.addcmul_(d, alpha)
        r.addcmul_(q, -alpha)
        if k % 50 == 49 and float(r.norm()) <= stop:
            break
        z = w * r
        rz, old = (r * z).sum(), rz
        d.mul_(rz / old).add_(z)
    return x if A.open else x - f * (x.sum() / cells)


def _exact_scene(s):
    p = _pressure(s["n"], s["h"], s["fluid"], s["wall"], s["rhs"])
    if "p0" in s and not any(s["wall"]):     # a closed box keeps the mean that it was given
        m = s["p0"][s["fluid"]].mean()
        p[s["fluid"]] += m
    return p


def exact(case, seed):
    kind = case["kind"]
    if kind == "amgpcg":
        n = case["n"]
        b = torch.from_numpy(_amg_rhs(n, seed).reshape(n + 2, n + 2)[1:-1, 1:-1].copy())
        k = torch.arange(1, n + 1, dtype=torch.float64)
        S = torch.sin(math.pi * torch.outer(k, k) / (n + 1)) * math.sqrt(2.0 / (n + 1))
        lam = 4.0 * torch.sin(0.5 * math.pi * k / (n + 1)) ** 2 * (n + 1) ** 2
        x = torch.zeros(n + 2, n + 2, dtype=torch.float64)
        x[1:-1, 1:-1] = S @ ((S @ b @ S) / (lam[:, None] + lam[None, :])) @ S
        return x.reshape(-1)
    if kind in ("batch", "serve"):
        return [_exact_scene(s) for s in _members(case, seed)]
    s = _scene(_dims(case), case["stretch"], case["balls"], case["slab"], case["walls"], case["warm"], seed, kind == "project")
    p = _exact_scene(s)
    if kind == "frame":
        return p.reshape(-1)
    if kind != "project":
        return p
    out, dim = [], len(s["n"])
    for a in range(dim):
        ax, na = dim - 1 - a, s["n"][a]
        f = s["vel"][a].clone()
        both = s["fluid"].narrow(ax, 0, na + 1) & s["fluid"].narrow(ax, 1, na + 1)
        f -= both * (DT / s["h"][a]) * (p.narrow(ax, 1, na + 1) - p.narrow(ax, 0, na + 1))
        out.append(f)
    return out + [p]
