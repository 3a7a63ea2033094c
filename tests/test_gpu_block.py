"""Smoothing visits of small levels as one launch each (csrc/block.hip) and pairs of iterations of
larger ones as one march (csrc/zmarch2.hpp): the same solve, bit for bit, as the oracle's and as the
marching launches that an explicit tile shape selects."""
import numpy as np
import pytest

import amrmg
import hierarchy as H
from oracle import Oracle

pytestmark = pytest.mark.gpu


def single(n, box, block, alpha, beta, lo=(0, 0, 0), bc=(1, 1, 1), hi_bc=(1, 1, 1)):
    dom = H.box(lo, [a + v - 1 for a, v in zip(lo, n)])
    return H.Hierarchy(dom, [H.domain_split(dom, box, block)], 1.0 / max(n), alpha, beta,
                       bc_type_lo=bc, bc_type_hi=hi_bc)


CASES = [
    # sizes that the 8^3 blocks cut raggedly, and one block only
    ("one_block", dict(n=(8, 8, 8), box=8, block=4, alpha=0.0, beta=1.0), 2, 0),
    ("ragged", dict(n=(20, 12, 36), box=12, block=4, alpha=0.4, beta=1.5, bc=(0, 1, 0)), 2, 0),
    # one, three and no iterations per visit, an origin off zero
    ("one", dict(n=(28, 20, 12), box=12, block=4, alpha=0.0, beta=1.0, lo=(-8, 4, 12)), 1, 0),
    ("three", dict(n=(28, 20, 12), box=12, block=4, alpha=0.2, beta=1.0, lo=(-8, 4, 12)), 3, 0),
    # the largest level of blocks with a coarser one below, and the first above
    ("last", dict(n=(128, 128, 64), box=64, block=16, alpha=0.1, beta=1.0), 2, 0),
    ("above", dict(n=(128, 128, 72), box=64, block=8, alpha=0.1, beta=1.0), 2, 0),
    # pairs of iterations: columns, chunks and pairs cut raggedly, an odd count, both tiles of FP32
    ("pairs", dict(n=(108, 92, 112), box=60, block=4, alpha=0.3, beta=1.2, bc=(0, 1, 1), hi_bc=(1, 0, 0)), 2, 0),
    ("pairs_odd", dict(n=(100, 108, 104), box=52, block=4, alpha=0.0, beta=1.0, lo=(-4, 8, 0)), 3, 0),
    ("pairs_single_precision", dict(n=(108, 92, 112), box=60, block=4, alpha=0.0, beta=1.0, bc=(0, 1, 1)), 2, 1),
    ("pairs_wide", dict(n=(236, 228, 236), box=120, block=4, alpha=0.2, beta=1.0), 2, 1),
    ("single_precision", dict(n=(20, 12, 36), box=12, block=4, alpha=0.0, beta=1.0, bc=(0, 1, 1)), 2, 1),
    ("single_precision_three", dict(n=(40, 24, 16), box=8, block=8, alpha=0.5, beta=1.0), 3, 1),
]


@pytest.mark.parametrize("name,spec,sweeps,precision", CASES, ids=[c[0] for c in CASES])
def test_block_visits_match_marching_launches(gpu_ctx, name, spec, sweeps, precision):
    h = single(**spec)
    rhs = H.bump_rhs(h, 1021)
    sp, rp = H.solver_params(pre=sweeps, post=sweeps, iterMax=4)
    runs = []
    for shape in (None, 16):
        g = amrmg.AMRMultiGrid(gpu_ctx, h, precision=precision)
        g.setSolverParameters(sp, rp)
        if shape is not None:
            g.set_relax_shape(shape, 0)
        g.set_field(g.RHS, rhs)
        hist, info = g.solve()
        runs.append((hist, g.get_field(g.PHI), info))
        if shape is None:                     # timed shapes keep the block visits
            g.tune_relax()
            again, _ = g.solve()
            np.testing.assert_array_equal(again, hist)
        g.close()
    assert runs[0][2] == runs[1][2]
    np.testing.assert_array_equal(runs[0][0], runs[1][0])
    np.testing.assert_array_equal(runs[0][1], runs[1][1])
    if precision == 0 and rhs.size < 1200000:
        o = Oracle(h)
        phi, hist, _ = o.solve(rhs, sp, rp)
        o.close()
        np.testing.assert_array_equal(runs[0][0], hist)
        np.testing.assert_array_equal(runs[0][1], phi)


def pieces(lo, hi, cuts):
    """The box lo..hi in boxes cut at `cuts` per direction."""
    ax = []
    for d in range(3):
        edges = [lo[d]] + [c for c in cuts[d] if lo[d] < c <= hi[d]] + [hi[d] + 1]
        ax.append([(edges[q], edges[q + 1] - 1) for q in range(len(edges) - 1)])
    return [((x[0], y[0], z[0]), (x[1], y[1], z[1])) for x in ax[0] for y in ax[1] for z in ax[2]]


def both_routes(ctx, h, rhs, sp, rp, precision, bottom_iterations=None):
    """(history, phi) with the default launches and with the marching launch per iteration."""
    runs = []
    for shape in (None, 16):
        g = amrmg.AMRMultiGrid(ctx, h, precision=precision)
        g.setSolverParameters(sp, rp)
        if bottom_iterations is not None:
            g.set_bottom_params(imax=bottom_iterations)
        if shape is not None:
            g.set_relax_shape(shape, 0)
        g.set_field(g.RHS, rhs)
        hist, _ = g.solve()
        runs.append((hist, g.get_field(g.PHI)))
        g.close()
    return runs


@pytest.mark.parametrize("n,precision", [
    ((107, 101, 99), 0),      # chunks of 12 planes
    ((149, 151, 143), 0),     # chunks of 16
    ((235, 231, 233), 0),     # chunks of 32
    ((107, 101, 99), 1),
    ((235, 231, 233), 1),     # the wider FP32 columns
])
def test_pair_march_odd_extents(gpu_ctx, n, precision):
    """Odd extents: each row's last pair is half outside the level.  The level has no coarser one, so a
    V-cycle is its five bottom iterations (a pair from zero, a pair, a single one; the Krylov solve
    ends before its first iteration)."""
    dom = H.box((0, 0, 0), [v - 1 for v in n])
    boxes = pieces(dom[0], dom[1], [[v // 2] for v in n])
    h = H.Hierarchy(dom, [boxes], 1.0 / max(n), 0.3, 1.1, bc_type_lo=(0, 1, 1), bc_type_hi=(1, 0, 1))
    rng = np.random.default_rng(8)
    phi, rhs = rng.standard_normal(h.total_cells()), rng.standard_normal(h.total_cells())
    sp, rp = H.solver_params(bottom=5, iterMax=1)
    a, b = both_routes(gpu_ctx, h, rhs, sp, rp, precision, bottom_iterations=0)
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])
    if precision == 0:
        runs = []
        for shape in (None, 16):
            g = amrmg.AMRMultiGrid(gpu_ctx, h)
            if shape is not None:
                g.set_relax_shape(shape, 0)
            runs.append(g.level_relax(0, phi, rhs, 3))
            g.close()
        np.testing.assert_array_equal(*runs)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("sweeps", [2, 3])
def test_pair_march_coarse_fine_faces(gpu_ctx, sweeps, precision):
    """A refined level of 106 x 104 x 102 cells on one wall, coarse-fine faces on its other sides."""
    dom = H.box((0, 0, 0), (63, 59, 59))
    lo, hi = (0, 8, 6), (105, 111, 107)
    h = H.Hierarchy(dom, [H.domain_split(dom, 32, 4), pieces(lo, hi, [[54], [60], [50]])], 1.0 / 64, 0.2, 1.1)
    rhs = H.bump_rhs(h, 1022)
    sp, rp = H.solver_params(pre=sweeps, post=sweeps, iterMax=3)
    a, b = both_routes(gpu_ctx, h, rhs, sp, rp, precision)
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])
