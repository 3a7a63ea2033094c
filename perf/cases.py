"""Timed cases: what programs that use this library have it do.

Every case is a dict of plain values.  ``kind`` says which public entry points it goes
through:

* ``solve``  one AMRMultiGrid solve to a 1e-10 relative residual from a zero guess: one
  level or AMR levels, FP64 or mixed precision, constant or variable coefficients, one or
  several components, any boundary condition, merged or per-box levels.
* ``heat``   one time step (AMRTGA or BackwardEuler) over an AMR hierarchy.
* ``batch``  many independent one-level Helmholtz problems solved together.
* ``serve``  a burst of requests of different sizes through the serving engine, host
  right-hand sides in, host solutions out.
* ``cycle``  a two-grid correction driven from the host through the operator handles
  (relax, residual, restrict, coarse relax, prolong, relax, apply, norm), as a program
  that keeps its own multigrid loop calls them.

A solver's fields live in HBM and stay there from solve to solve; a program reads one out
when it wants it on the host.  ``run`` therefore returns such a field as a ``Fields``
entry, which is read out when it is looked at, as a GPU tensor would be.  Where an entry
point itself takes and gives host data (serve), the copies are part of the pass.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "chombo_3.2_amd"))

import amrmg  # noqa: E402
import hierarchy as H  # noqa: E402
import levelops as LO  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"
EPS = 1e-10


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest calls: a host-driven two-grid cycle on a block of 31 thousand cells
        dict(name="cycle_24x40x32", kind="cycle", nx=24, ny=40, nz=32, box=32, alpha=0.0, beta=1.0),
        # the same on a level of 6.9 million cells, extents that no tile divides
        dict(name="cycle_216x160x200", kind="cycle", nx=216, ny=160, nz=200, box=64, alpha=0.3, beta=1.0),
        # the single-level benchmark: 64^3 Poisson in 32^3 boxes
        dict(name="solve_64", kind="solve", nx=64, ny=64, nz=64, box=32, block=8, fracs=""),
        # a ragged domain (bottom 30x22x26), Helmholtz, walls and insulated faces
        dict(name="solve_120x88x104", kind="solve", nx=120, ny=88, nz=104, box=40, block=8, fracs="", alpha=0.7,
             beta=1.3, bc="mixed"),
        # the flagship: 3-level AMR Poisson, base 256^3, FP64, tiles tuned beforehand
        dict(name="amr3_256", kind="solve", nx=256, ny=256, nz=256, box=64, block=8, fracs="0.25,0.06", tune=True),
        # the same in mixed precision
        dict(name="amr3_256_mixed", kind="solve", nx=256, ny=256, nz=256, box=64, block=8, fracs="0.25,0.06",
             tune=True, mixed=True),
        # variable coefficients on an AMR hierarchy, FP64
        dict(name="amr3_128_vc", kind="solve", nx=128, ny=128, nz=128, box=64, block=8, fracs="0.25,0.06", vc=True),
        # a refined region that is no rectangle (per-box storage), ratio 4, one periodic direction
        dict(name="amr2_64_notched_r4", kind="solve", nx=64, ny=64, nz=96, box=32, block=8, fracs="0.15", ratio=4,
             notch=True, bc="channel"),
        # a velocity-like field of three components on two levels
        dict(name="amr2_96_ncomp3", kind="solve", nx=96, ny=96, nz=96, box=48, block=8, fracs="0.2", ncomp=3),
        # time stepping: AMRTGA over two levels
        dict(name="heat_tga_128", kind="heat", nx=128, ny=128, nz=128, box=64, block=8, fracs="0.2", scheme="tga"),
        # many small problems at once, sizes 16..128 log-uniform, mixed precision
        dict(name="batch_96_mixed", kind="batch", count=96, nmin=16, nmax=128, mixed=True, lanes=3),
        # requests of 1-2 levels through the serving engine
        dict(name="serve_24", kind="serve", count=24, bases="32,64,128", slots=8),
    ]


def draw(rng):
    """One more case of these ranges, no larger than the listed ones."""
    def size(lo, hi, step):
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return int(max(lo, min(hi, step * round(v / step))))

    def ab():
        return (0.0, 1.0) if rng.random() < 0.5 else (round(rng.uniform(0.0, 1.0), 3), round(rng.uniform(0.5, 2.0), 3))

    kind = rng.choice(["cycle", "solve", "solve", "amr", "amr", "heat", "batch", "serve"])
    if kind == "cycle":
        a, b = ab()
        return dict(kind="cycle", nx=size(16, 256, 4), ny=size(16, 256, 4), nz=size(16, 256, 4),
                    box=rng.choice([32, 40, 64]), alpha=a, beta=b)
    if kind == "solve":
        a, b = ab()
        return dict(kind="solve", nx=size(16, 192, 8), ny=size(16, 192, 8), nz=size(16, 192, 8),
                    box=rng.choice([24, 32, 64]), block=8, fracs="", alpha=a, beta=b,
                    bc=rng.choice(["walls", "mixed"]), mixed=rng.random() < 0.4)
    if kind == "amr":
        what = rng.choice(["plain", "plain", "vc", "notch", "ncomp", "ratio4"])
        c = dict(kind="solve", nx=size(32, 128, 8), ny=size(32, 128, 8), nz=size(32, 128, 8),
                 box=rng.choice([32, 64]), block=8,
                 fracs="%.3f" % rng.uniform(0.05, 0.25) + (",%.3f" % rng.uniform(0.01, 0.04) if rng.random() < 0.4 else ""))
        if what == "vc":
            c.update(vc=True, mixed=rng.random() < 0.5)
        elif what == "notch":
            c.update(notch=True, bc=rng.choice(["walls", "channel"]), fracs=c["fracs"].split(",")[0])
        elif what == "ncomp":
            c.update(ncomp=rng.choice([2, 3]), nx=min(c["nx"], 96), ny=min(c["ny"], 96), nz=min(c["nz"], 96))
        elif what == "ratio4":
            c.update(ratio=4, fracs="%.3f" % rng.uniform(0.02, 0.06))
        else:
            c.update(mixed=rng.random() < 0.5, tune=rng.random() < 0.5)
        return c
    if kind == "heat":
        return dict(kind="heat", nx=size(48, 128, 8), ny=size(48, 128, 8), nz=size(48, 128, 8), box=64, block=8,
                    fracs="%.3f" % rng.uniform(0.05, 0.25), scheme=rng.choice(["tga", "be"]))
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(8, 96), nmin=16, nmax=rng.choice([48, 96, 128]),
                    mixed=rng.random() < 0.5, lanes=rng.choice([1, 2, 3]), tree=rng.random() < 0.3)
    return dict(kind="serve", count=rng.randint(4, 32), bases=rng.choice(["32,64", "32,64,128"]),
                slots=rng.choice([2, 4, 8]), mixed=rng.random() < 0.3)


# ---------------------------------------------------------------------------
# layouts and right-hand sides
# ---------------------------------------------------------------------------
BCS = {"walls": ((1, 1, 1), (1, 1, 1)), "mixed": ((1, 0, 1), (0, 1, 1)), "channel": ((3, 1, 1), (3, 1, 1))}


def region(n, frac, block, inside):
    """Centred box of about `frac` of a domain of extents n, snapped to the blocking factor and
    at least one block inside the box `inside`."""
    lo, hi = [], []
    for d in range(3):
        side = max(block, block * int(round(n[d] * frac ** (1.0 / 3.0) / block)))
        a = block * (((n[d] - side) // 2) // block)
        lo.append(max(a, inside[0][d] + block))
        hi.append(min(a + side - 1, inside[1][d] - block))
        if hi[d] < lo[d]:
            lo[d], hi[d] = a, a + block - 1
    return H.box(lo, hi)


def hierarchy_of(c):
    n = (c["nx"], c["ny"], c["nz"])
    lo, hi = BCS[c.get("bc", "walls")]
    dom = H.box((0, 0, 0), [v - 1 for v in n])
    box, block, r = c["box"], c.get("block", 8), int(c.get("ratio", 2))
    levels, ratios, ext, inside = [H.domain_split(dom, box, block)], [], n, dom
    for f in [float(v) for v in c.get("fracs", "").split(",") if v]:
        inside = H.box_refine(region(ext, f, block, inside), r)
        side = max(H.box_shape(inside))
        boxes = H.domain_split(inside, min(box, max(16, side // 16 * 8)) if c.get("notch") else box, block)
        if c.get("notch") and len(boxes) > 1:
            boxes = boxes[:-1]  # the box at the high corner is not refined
        levels.append(boxes)
        ratios.append(r)
        ext = [v * r for v in ext]
    return H.Hierarchy(dom, levels, 1.0 / max(n), c.get("alpha", 0.0), c.get("beta", 1.0), bc_type_lo=lo, bc_type_hi=hi,
                       ratios=tuple(ratios) if r != 2 else None)


def bumps(h, seed, ncomp=1):
    """Gaussian bumps (as the benchmark's right-hand side), box by box, each box component
    by component; formed on the GPU in FP64."""
    rng = np.random.default_rng(seed)
    top = h.dx0 * np.asarray(H.box_shape(h.domain))
    nb = 3 * ncomp
    cs, ws, ss = rng.uniform(0.35, 0.65, (nb, 3)) * top, rng.uniform(5e-3, 2e-2, nb), rng.uniform(1.0, 3.0, nb)
    out = torch.empty(h.total_cells() * ncomp, dtype=torch.float64, device=DEV)
    o = 0
    for lev in range(h.nlev):
        dx = h.dx(lev)
        for lo, hi in h.levels[lev]:
            xs = [(torch.arange(lo[d], hi[d] + 1, dtype=torch.float64, device=DEV) + 0.5) * dx for d in range(3)]
            m = len(xs[0]) * len(xs[1]) * len(xs[2])
            for q in range(ncomp):
                v = 0.0
                for b in range(q, nb, ncomp):
                    e = [torch.exp(-((xs[d] - cs[b, d]) ** 2) / ws[b]) for d in range(3)]
                    v = v + ss[b] * e[2][:, None, None] * e[1][None, :, None] * e[0][None, None, :]
                out[o:o + m] = v.reshape(-1)
                o += m
    return out.cpu().numpy()


def waves(n, seed):
    """sin waves and seeded noise on one n^3 level, as a dense [k, j, i] array."""
    g = torch.Generator(device="cpu").manual_seed(int(seed))
    k = torch.randint(1, 4, (3,), generator=g)
    x = [(torch.arange(v, dtype=torch.float64) + 0.5) / max(n) for v in n]
    s = [torch.sin(2 * math.pi * int(k[d]) * x[d]) for d in range(3)]
    noise = torch.randn(n[2], n[1], n[0], dtype=torch.float64, generator=g)
    return s[2][:, None, None] * s[1][None, :, None] * s[0][None, None, :] + 1e-3 * noise


def pack(h, dense):
    """A dense [k, j, i] array over level 0, box by box in Fortran order."""
    a = dense.numpy() if isinstance(dense, torch.Tensor) else dense
    parts = [a[lo[2]:hi[2] + 1, lo[1]:hi[1] + 1, lo[0]:hi[0] + 1].reshape(-1) for lo, hi in h.levels[0]]
    return np.concatenate(parts)


def batch_specs(c, seed):
    rng = np.random.default_rng(1004 + 31 * c["count"] + c["nmax"])  # sizes and coefficients belong to the case
    out = []
    for q in range(c["count"]):
        n = int(8 * round(math.exp(rng.uniform(math.log(c["nmin"]), math.log(c["nmax"]))) / 8))
        n = max(8, min(c["nmax"], n))
        dom = H.box((0, 0, 0), (n - 1,) * 3)
        h = H.Hierarchy(dom, [H.domain_split(dom, 64, 8)], 1.0 / n, float(rng.uniform(0.0, 1.0)),
                        float(rng.uniform(0.5, 2.0)))
        out.append((h, waves((n, n, n), seed * 100003 + q)))
    return out


def serve_specs(c, seed):
    rng = np.random.default_rng(1005 + 17 * c["count"])
    bases = [int(v) for v in c["bases"].split(",")]
    out = []
    for q in range(c["count"]):
        n, two, f = int(rng.choice(bases)), bool(rng.integers(0, 2)), float(rng.uniform(0.05, 0.25))
        h = hierarchy_of(dict(nx=n, ny=n, nz=n, box=64, block=8, fracs="%.3f" % f if two else ""))
        out.append((h, bumps(h, seed * 1009 + q)))
    return out


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------
_ctx = None


def context():
    global _ctx
    if _ctx is None:
        _ctx = amrmg.Context(0)
    return _ctx


class Fields(dict):
    """Device-resident results by name; a field is read out when it is looked at."""

    def __init__(self, state, read, **values):
        super().__init__(values)
        self.state = state  # the handles live as long as what can still be read from them
        self.read = read
        for k in read:
            self[k] = None

    def __getitem__(self, k):
        return self.read[k]() if k in self.read else super().__getitem__(k)


class State:
    def __init__(self, case, **kw):
        self.case = case
        self.__dict__.update(kw)


class CycleState(State):
    """Operator handles of a two-grid cycle; handles are given back with the state."""

    def __del__(self):
        try:
            for x in self.fields + [self.child, self.op, self.level]:
                x.close()
        except Exception:
            pass


def params():
    return H.solver_params(eps=EPS, hang=1e-15, iterMax=100)


def prepare(case, seed):
    c, ctx, kind = case, context(), case["kind"]
    if kind == "cycle":
        n = (c["nx"], c["ny"], c["nz"])
        dom = H.box((0, 0, 0), [v - 1 for v in n])
        h = H.Hierarchy(dom, [H.domain_split(dom, c["box"], 4)], 1.0 / max(n))
        level = LO.Level(ctx, h.levels[0], dom)
        op = LO.AMRPoissonOp(level, h.dx0, alpha=c["alpha"], beta=c["beta"])
        child = op.createCoarser()
        f = {k: LO.Field(level) for k in ("phi", "rhs", "res", "lap")}
        f.update({k: LO.Field(child.level) for k in ("resC", "eC")})
        f["rhs"].upload(pack(h, waves(n, seed)))
        return CycleState(c, level=level, op=op, child=child, f=f, fields=list(f.values()))
    if kind == "batch":
        specs = batch_specs(c, seed)
        b = amrmg.BatchSolver(ctx, [h for h, _ in specs], precision=int(c.get("mixed", False)), lanes=c["lanes"])
        b.setSolverParameters(*params())
        if c.get("tree"):
            b.set_reduction_order(1)
        for q, (h, w) in enumerate(specs):
            b.set_rhs(q, pack(h, w))
        return State(c, batch=b)
    if kind == "serve":
        sp, rp = params()
        e = amrmg.ServeEngine(0, slots=c["slots"], budget_bytes=64 << 30, precision=int(c.get("mixed", False)),
                              sparams=sp, rparams=rp, max_large=max(1, c["slots"] // 2), large_cells=1 << 21)
        return State(c, engine=e, reqs=serve_specs(c, seed))
    h = hierarchy_of(c)
    nc = int(c.get("ncomp", 1))
    s = amrmg.AMRMultiGrid(ctx, h, precision=int(c.get("mixed", False)), ncomp=nc)
    s.setSolverParameters(*params())
    rhs = bumps(h, seed, nc)
    if kind == "heat":
        heat = amrmg.HeatSolver(s, c["scheme"])
        heat.set_source(rhs)
        s.set_field(s.PHI, 0.05 * bumps(h, seed + 7919))
        return State(c, solver=s, heat=heat)
    if c.get("vc"):
        s.set_vc_coefs(*H.vc_coefficients(h, seed=7, contrast=4.0))
    s.set_field(s.RHS, rhs)
    if c.get("tune"):
        s.tune_relax()
    return State(c, solver=s)


def run(state):
    kind = state.case["kind"]
    if kind == "solve":
        s = state.solver
        hist, _ = s.solve()
        return Fields(state, {"phi": lambda: s.get_field(s.PHI)}, history=np.pad(hist, (0, 101 - len(hist))))
    if kind == "heat":
        s = state.solver
        state.heat.step(1e-3)
        return Fields(state, {"phi": lambda: s.get_field(s.PHI)})
    if kind == "batch":
        b = state.batch
        b.solve()
        return Fields(state, {"phi": lambda: np.concatenate([b.get_phi(q) for q in range(b.n)])})
    if kind == "serve":
        e = state.engine
        ids = [e.submit(h, r) for h, r in state.reqs]
        return [e.wait(i)["phi"] for i in ids]
    op, child, f = state.op, state.child, state.f
    op.setToZero(f["phi"])
    op.relax(f["phi"], f["rhs"], 2)
    op.residual(f["res"], f["phi"], f["rhs"], True)
    op.restrictResidual(f["resC"], f["phi"], f["rhs"])
    child.setToZero(f["eC"])
    child.relax(f["eC"], f["resC"], 4)
    op.prolongIncrement(f["phi"], f["eC"])
    op.relax(f["phi"], f["rhs"], 2)
    op.applyOp(f["lap"], f["phi"], True)
    norm = op.norm(f["res"], 0)
    return Fields(state, {k: f[k].download for k in ("phi", "res", "lap", "resC")}, norm=norm)


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def mg_cells(cells, depths):
    return sum(cells / 8.0 ** d for d in range(depths))


def cycle_work(c, h):
    """Bytes and flops of one V-cycle of a hierarchy: on every level the two smoothing
    visits read the correction and the right-hand side and write the correction once,
    the residual reads two fields and writes one, the update reads two and writes one
    (variable coefficients: four more fields per visit and residual)."""
    cells = sum(h.cells(l) for l in range(1, h.nlev)) + mg_cells(h.cells(0), 4)
    nc = int(c.get("ncomp", 1))
    size = 4.0 if c.get("mixed") else 8.0
    vc = 4.0 if c.get("vc") else 0.0
    return nc * cells * (2 * (3 + vc) * size + (3 + vc) * size + 24.0), nc * cells * (4 * 11 + 10 + 2)


def work(case):
    c, kind = case, case["kind"]
    if kind == "cycle":
        n = float(c["nx"] * c["ny"] * c["nz"])
        # two smoothing visits, residual, restriction, prolongation, apply, norm; the coarse visit
        return {"bytes": n * (16 + 24 + 24 + 17 + 17 + 16 + 8) + n / 8 * 24, "flops": n * (4 * 11 + 3 * 10) + n / 8 * 44}
    if kind == "batch":
        rng = np.random.default_rng(1004 + 31 * c["count"] + c["nmax"])
        cells = 0.0
        for _ in range(c["count"]):
            n = int(8 * round(math.exp(rng.uniform(math.log(c["nmin"]), math.log(c["nmax"]))) / 8))
            cells += max(8, min(c["nmax"], n)) ** 3
            rng.uniform(0.0, 1.0), rng.uniform(0.5, 2.0)
        size = 4.0 if c.get("mixed") else 8.0
        b = 10 * mg_cells(cells, 4) * (9 * size + 24)
        return {"bytes": b, "flops": 10 * mg_cells(cells, 4) * 56}
    if kind == "serve":
        rng = np.random.default_rng(1005 + 17 * c["count"])
        bases = [int(v) for v in c["bases"].split(",")]
        b = f = 0.0
        for _ in range(c["count"]):
            n, two, fr = int(rng.choice(bases)), bool(rng.integers(0, 2)), float(rng.uniform(0.05, 0.25))
            h = hierarchy_of(dict(nx=n, ny=n, nz=n, box=64, block=8, fracs="%.3f" % fr if two else ""))
            x, y = cycle_work(c, h)
            b, f = b + 11 * x + 16.0 * h.total_cells(), f + 11 * y
        return {"bytes": b, "flops": f}
    h = hierarchy_of(c)
    b, f = cycle_work(c, h)
    cycles = {"heat": 20 if c.get("scheme") == "tga" else 11}.get(kind, 12 if h.nlev > 1 else 10)
    return {"bytes": cycles * b, "flops": cycles * f}


def tolerance(case):
    """FP64 operations against their sums in another order: at most 7e-15 (the operator's
    1/dx^2 cancellation).  Solves stop at a 1e-10 relative residual: at most 4.4e-11 from the
    direct solution, in FP64 and in mixed precision, so another correct solver's result
    differs by that much."""
    if case["kind"] == "cycle":
        return {"rel": 3e-14, "max": 1e-12}
    return {"rel": 2e-10, "max": 8e-9}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def line(n, lo, hi):
    """1-D second difference of n cells with the faces' homogeneous ghosts (0 Neumann, 1
    Dirichlet, 3 periodic)."""
    a = torch.zeros(n, n, dtype=torch.float64)
    i = torch.arange(n)
    a[i, i] = -2.0
    a[i[:-1], i[1:]] = 1.0
    a[i[1:], i[:-1]] = 1.0
    if lo == 3:
        a[0, n - 1] += 1.0
        a[n - 1, 0] += 1.0
    else:
        a[0, 0] += -1.0 if lo == 1 else 1.0
        a[n - 1, n - 1] += -1.0 if hi == 1 else 1.0
    return a


def direct(h, rhs):
    """Solution of (alpha + beta lap) phi = rhs on one level by the eigenvectors of each direction."""
    v, w = [], []
    for d in range(3):
        n = h.domain[1][d] + 1
        e, q = torch.linalg.eigh(line(n, h.bc_type_lo[d], h.bc_type_hi[d]).to(DEV))
        v.append(q)
        w.append(e / h.dx0 ** 2)
    x = rhs.to(DEV)
    turn = lambda x, m: torch.tensordot(torch.tensordot(torch.tensordot(  # noqa: E731
        x, m[2], ([0], [0])), m[1], ([0], [0])), m[0], ([0], [0]))
    x = turn(x, v)
    x = x / (h.alpha + h.beta * (w[2][:, None, None] + w[1][None, :, None] + w[0][None, None, :]))
    return turn(x, [m.T.contiguous() for m in v]).cpu()


def unpack(h, data):
    n = H.box_shape(h.domain)
    a = np.empty((n[2], n[1], n[0]))
    o = 0
    for lo, hi in h.levels[0]:
        s = (hi[2] - lo[2] + 1, hi[1] - lo[1] + 1, hi[0] - lo[0] + 1)
        m = s[0] * s[1] * s[2]
        a[lo[2]:hi[2] + 1, lo[1]:hi[1] + 1, lo[0]:hi[0] + 1] = data[o:o + m].reshape(s)
        o += m
    return torch.from_numpy(a)


def laplacian(x, dx):
    """7-point Laplacian of a dense level with homogeneous linear Dirichlet faces."""
    s = -6.0 * x
    for d in range(3):
        n = x.shape[d]
        g = torch.cat([-x.narrow(d, 0, 1), x, -x.narrow(d, n - 1, 1)], d)
        s = s + g.narrow(d, 0, n) + g.narrow(d, 2, n)
    return s / (dx * dx)


def smooth(x, r, dx, alpha, beta, times):
    n = x.shape
    par = sum(torch.arange(n[d], device=x.device).reshape([-1 if q == d else 1 for q in range(3)]) for d in range(3)) % 2
    lam = 1.0 / (alpha - beta * 6.0 / (dx * dx))
    for _ in range(times):
        for colour in (0, 1):
            x = torch.where(par == colour, x + lam * (r - alpha * x - beta * laplacian(x, dx)), x)
    return x


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "cycle":
        n = (c["nx"], c["ny"], c["nz"])
        dom = H.box((0, 0, 0), [v - 1 for v in n])
        h = H.Hierarchy(dom, [H.domain_split(dom, c["box"], 4)], 1.0 / max(n))
        hc = H.Hierarchy(H.box_coarsen(dom, 2), [[H.box_coarsen(b, 2) for b in h.levels[0]]], 2 * h.dx0)
        a, b, dx = c["alpha"], c["beta"], h.dx0
        r = waves(n, seed).to(DEV)
        x = smooth(torch.zeros_like(r), r, dx, a, b, 2)
        res = r - a * x - b * laplacian(x, dx)
        rc = res.reshape(n[2] // 2, 2, n[1] // 2, 2, n[0] // 2, 2).mean((1, 3, 5))
        e = smooth(torch.zeros_like(rc), rc, 2 * dx, a, b, 4)
        x = x + e.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)
        x = smooth(x, r, dx, a, b, 2)
        lap = a * x + b * laplacian(x, dx)
        return {"phi": pack(h, x.cpu()), "res": pack(h, res.cpu()), "lap": pack(h, lap.cpu()), "resC": pack(hc, rc.cpu()),
                "norm": float(res.abs().max())}
    if kind == "batch":
        return {"phi": np.concatenate([pack(h, direct(h, w)) for h, w in batch_specs(c, seed)])}
    if kind == "serve":
        return [pack(h, direct(h, unpack(h, r))) if h.nlev == 1 else None for h, r in serve_specs(c, seed)]
    # a composite AMR or variable-coefficient system has no direct form here: its plain
    # Krylov solve takes minutes
    if kind == "heat" or c.get("fracs") or c.get("vc") or c.get("ncomp", 1) > 1:
        return None
    h = hierarchy_of(c)
    return {"phi": pack(h, direct(h, unpack(h, bumps(h, seed)))), "history": None}
