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
