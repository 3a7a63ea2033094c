"""The z march of the variable-coefficient relaxation (csrc/vczmarch.hpp) where its pairs, columns and
chunks end raggedly: level relaxations and solves equal the tile shape 0 launches bit for bit."""
import numpy as np
import pytest

import amrmg
import hierarchy as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,bc", [
    ((1, 3, 2), (1, 1, 1)),
    ((37, 29, 23), (0, 1, 1)),          # odd rows: the last pair is half outside
    ((64, 20, 40), (1, 0, 1)),          # whole columns, faces of every kind
    ((98, 62, 90), (1, 1, 0)),          # chunks of 8 planes, the last one short
])
def test_vc_march_matches_tile_launches(gpu_ctx, n, bc, precision):
    dom = H.box((0, 0, 0), [v - 1 for v in n])
    h = H.Hierarchy(dom, [[dom]], 1.0 / max(n), 0.7, 1.3, bc_type_lo=bc, bc_type_hi=(1, 1, 1))
    cells = int(np.prod(n))
    runs = []
    for shape in (-1, 0):
        g = amrmg.AMRMultiGrid(gpu_ctx, h, precision=precision)
        g.set_vc_coefs(*H.vc_coefficients(h, seed=5, contrast=4.0))
        g.set_vc_relax_shape(shape)
        rng = np.random.default_rng(3)
        p, r = rng.standard_normal(cells), rng.standard_normal(cells)
        lv = g.level_relax(0, p, r, 3)
        run = [lv]
        if cells < 60000:                # the bottom level of the largest is far from small
            sp, rp = H.solver_params(iterMax=3)
            g.setSolverParameters(sp, rp)
            g.set_field(g.RHS, r)
            hist, _ = g.solve()
            run += [hist, g.get_field(g.PHI)]
        runs.append(run)
        g.close()
    for x, y in zip(*runs):
        np.testing.assert_array_equal(x, y)
