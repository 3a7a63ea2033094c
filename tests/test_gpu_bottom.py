"""The device bottom solve at the sizes where its tables change form: against the
host-driven BiCGStab of the same level (the same operations and reduction orders, so the
correction is bitwise the same and the iteration counts agree)."""
import numpy as np
import pytest

import hierarchy as H

pytestmark = pytest.mark.gpu


def _level(n, cuts, alpha, beta, bc):
    """One level of n cells cut into boxes at `cuts` per direction (odd extents: no coarser level)."""
    ax = []
    for d in range(3):
        edges = [0] + [c for c in cuts[d] if 0 < c < n[d]] + [n[d]]
        ax.append([(edges[q], edges[q + 1] - 1) for q in range(len(edges) - 1)])
    boxes = [((x[0], y[0], z[0]), (x[1], y[1], z[1])) for x in ax[0] for y in ax[1] for z in ax[2]]
    return H.Hierarchy(H.box((0, 0, 0), [v - 1 for v in n]), [boxes], 1.0 / max(n), alpha, beta,
                       bc_type_lo=bc[0], bc_type_hi=bc[1])


WALLS = ((1, 1, 1), (1, 1, 1))
MIXED = ((1, 0, 1), (0, 1, 0))


@pytest.mark.parametrize("n,cuts,ab,bc", [
    ((1, 1, 3), ([], [], []), (0.5, 1.0), WALLS),                      # one cell wide
    ((4, 5, 3), ([], [2], []), (0.0, 1.0), WALLS),                     # one wave
    ((7, 4, 9), ([3], [], [5]), (0.7, 1.3), MIXED),                    # odd rows, 144 slots
    ((8, 8, 9), ([], [], []), (0.0, 1.0), MIXED),                      # 288 slots: 1024 threads, inner entries
    ((13, 11, 16), ([5], [4], [8]), (0.2, 0.9), WALLS),                # 1232 slots
    ((27, 26, 25), ([9], [13], [8, 16]), (0.7, 1.3), MIXED),           # 9100 slots: both colours in LDS
    ((29, 31, 30), ([15], [16], [14]), (0.3, 1.1), WALLS),             # 13950 slots: one colour, three stages
    ((32, 31, 33), ([], [], []), (0.9, 0.6), MIXED),                   # 16368 slots, one box
    ((33, 32, 33), ([16], [16], [16]), (0.9, 0.6), WALLS),             # past the slot tables: the general kernel
])
def test_device_bottom_equals_host_bicgstab(gpu_ctx, n, cuts, ab, bc):
    import amrmg
    h = _level(n, cuts, ab[0], ab[1], bc)
    s = amrmg.AMRMultiGrid(gpu_ctx, h)
    rng = np.random.default_rng(sum(n))
    res = rng.standard_normal(h.total_cells())
    corr = 0.1 * rng.standard_normal(h.total_cells())
    metric = float(np.sqrt((res ** 2).sum()))
    want, _, iters = s.bottom_solve(corr, res, 2, metric, 1e-10)
    got, _, dev_iters = s.bottom_solve(corr, res, 2, metric, 1e-10, device=True)
    s.close()
    assert dev_iters == iters
    assert np.array_equal(got, want)


PERIODIC = ((3, 1, 3), (3, 0, 3))
CHANNEL = ((1, 3, 1), (0, 3, 1))


@pytest.mark.parametrize("n,cuts,ab,bc,nc", [
    ((18, 14, 22), ([10], [], [12]), (0.5, 0.9), PERIODIC, 1),           # per box, both colours in LDS
    ((30, 30, 30), ([14], [16], []), (0.6, 1.1), PERIODIC, 1),           # per box, one colour
    ((14, 10, 6), ([], [4], []), (0.3, 1.2), CHANNEL, 2),                # components of per-box levels
    ((20, 21, 19), ([9], [], [8]), (0.7, 1.3), MIXED, 3),                # 11970 slots of three components
])
def test_device_bottom_periodic_and_components(gpu_ctx, n, cuts, ab, bc, nc):
    """Levels that the bottom entry point does not take (per box or several components), through whole
    solves: no coarser level, so a V-cycle is the bottom from zero.  The oracle's history, solution and
    iteration counts, bit for bit."""
    import amrmg
    from helpers import comps_pack
    from oracle import Oracle
    h = _level(n, cuts, ab[0], ab[1], bc)
    rng = np.random.default_rng(sum(n))
    rhs = comps_pack(h, [rng.standard_normal(h.total_cells()) for _ in range(nc)])
    sp, rp = H.solver_params(iterMax=3)
    g, o = amrmg.AMRMultiGrid(gpu_ctx, h, ncomp=nc), Oracle(h)
    if nc > 1:
        o.set_ncomp(nc)
    assert g.mg_depths == 1
    g.setSolverParameters(sp, rp)
    g.set_field(g.RHS, rhs)
    hist, info = g.solve()
    phi_o, hist_o, info_o = o.solve(rhs, sp, rp)
    phi = g.get_field(g.PHI)
    g.close()
    o.close()
    assert info["iterations"] == info_o["iterations"] and info["exit_status"] == info_o["exit_status"]
    np.testing.assert_array_equal(hist, hist_o)
    np.testing.assert_array_equal(phi, phi_o)


def _relaxed_from_zero(n, rhs, h, lo, hi, its, dtype):
    """`its` red-black iterations of a zero field with homogeneous faces, in `dtype`, one rounding per
    operation in the kernels' order."""
    c = lambda v: dtype(v)  # noqa: E731
    dxinv = 1.0 / (h.dx0 * h.dx0)
    sum_b = 0.0
    for _ in range(3):
        sum_b += 2.0 * dxinv
    lam = c(-1.0 / (h.alpha - h.beta * sum_b))
    x = np.zeros(n, dtype=dtype)
    par = np.add.outer(np.add.outer(np.arange(n[0]), np.arange(n[1])), np.arange(n[2])) % 2
    for it in range(2 * its):
        nb = []
        for d in range(3):
            first, last = np.take(x, [0], d), np.take(x, [-1], d)
            g = np.concatenate([-first if lo[d] else first, x, -last if hi[d] else last], d)
            nb += [np.take(g, range(2, n[d] + 2), d), np.take(g, range(0, n[d]), d)]
        s = nb[0] + nb[1] + nb[2] + nb[3] + nb[4] + nb[5]
        lap = (s - c(6.0) * x) * c(dxinv)
        x = np.where(par == it % 2, x + lam * ((c(h.alpha) * x + c(h.beta) * lap) - rhs), x)
    return x


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [(4, 5, 3), (13, 11, 16), (27, 26, 25), (29, 31, 30), (32, 31, 33)])
def test_bottom_relaxation_from_zero(gpu_ctx, n, precision):
    """The relaxations with which the bottom starts, in the V-cycle's precision (one V-cycle on a level
    without a coarser one; the Krylov solve ends before its first iteration and adds zero), where both
    colours are in LDS and where one is."""
    import amrmg
    dtype = (np.float64, np.float32)[precision]
    h = _level(n, ([], [], []), 0.7, 1.3, MIXED)
    rhs = np.random.default_rng(sum(n)).standard_normal(h.total_cells())
    g = amrmg.AMRMultiGrid(gpu_ctx, h, precision=precision)
    assert g.mg_depths == 1
    sp, rp = H.solver_params(bottom=3, iterMax=1)
    g.setSolverParameters(sp, rp)
    g.set_bottom_params(imax=0)
    g.set_field(g.RHS, rhs)
    g.solve()
    got = g.get_field(g.PHI).reshape(n, order="F")
    g.close()
    want = _relaxed_from_zero(n, rhs.reshape(n, order="F").astype(dtype), h, MIXED[0], MIXED[1], 3, dtype)
    assert want.dtype == dtype
    np.testing.assert_array_equal(got, want.astype(np.float64))
