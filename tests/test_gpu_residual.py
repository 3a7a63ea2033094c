"""The residual march (k_residual_z) where its pairs, columns and chunks end raggedly: residuals and
their max-norm equal the oracle's bit for bit."""
import numpy as np
import pytest

import amrmg
import hierarchy as H
from oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 2), (3, 5, 9), (37, 29, 23), (64, 4, 8), (66, 9, 17)])
def test_residual_and_norm_bitwise(gpu_ctx, n):
    dom = H.box((0, 0, 0), [v - 1 for v in n])
    h = H.Hierarchy(dom, [[dom]], 1.0 / max(n), 0.7, 1.3, bc_type_lo=(1, 0, 1), bc_type_hi=(0, 1, 1))
    rng = np.random.default_rng(11)
    phi, rhs = rng.standard_normal(int(np.prod(n))), rng.standard_normal(int(np.prod(n)))
    g, o = amrmg.AMRMultiGrid(gpu_ctx, h), Oracle(h)
    for homog in (False, True):
        np.testing.assert_array_equal(g.level_residual(0, phi, rhs, homog), o.level_residual(0, phi, rhs, homog))
    sp, rp = H.solver_params(iterMax=0)
    g.setSolverParameters(sp, rp)
    g.set_field(g.RHS, rhs)
    hist, _ = g.solve()
    assert hist[0] == np.abs(rhs).max()     # the residual of a zero field
    g.close()
    o.close()
