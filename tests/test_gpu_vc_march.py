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
    ((98, 62, 90), (1, 1, 0)),          # chunks of 4 planes, the last one short
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


# Levels of at least 512 chunks of 8 planes keep that length: the march's slots wrap around there, and
# the operands it carries from step to step pass the loop's back edge.
def test_vc_march_chunks_of_eight_odd(gpu_ctx):
    n = (131, 123, 133)                     # 5 x 13 x 17 chunks, the last one of 5 planes
    dom = H.box((0, 0, 0), [v - 1 for v in n])
    h = H.Hierarchy(dom, [[dom]], 1.0 / max(n), 0.7, 1.3, bc_type_lo=(0, 1, 1), bc_type_hi=(1, 1, 0))
    rng = np.random.default_rng(4)
    p, r = rng.standard_normal(h.total_cells()), rng.standard_normal(h.total_cells())
    runs = []
    for shape in (-1, 0):
        g = amrmg.AMRMultiGrid(gpu_ctx, h)
        g.set_vc_coefs(*H.vc_coefficients(h, seed=5, contrast=4.0))
        g.set_vc_relax_shape(shape)
        runs.append(g.level_relax(0, p, r, 3))
        g.close()
    np.testing.assert_array_equal(*runs)


@pytest.mark.parametrize("precision", [0, 1])
def test_vc_march_chunks_of_eight_solve(gpu_ctx, precision):
    """V-cycles: from zero, in both precisions; the bottom (70 x 62 x 66) takes few BiCGStab iterations."""
    n = (140, 124, 132)                     # 5 x 13 x 17 chunks, the last one of 4 planes
    dom = H.box((0, 0, 0), [v - 1 for v in n])
    h = H.Hierarchy(dom, [H.domain_split(dom, 72, 4)], 1.0 / max(n), 0.7, 1.3, bc_type_lo=(1, 0, 1))
    rng = np.random.default_rng(6)
    rhs = rng.standard_normal(h.total_cells())
    sp, rp = H.solver_params(iterMax=2)
    runs = []
    for shape in (-1, 0):
        g = amrmg.AMRMultiGrid(gpu_ctx, h, precision=precision)
        g.set_vc_coefs(*H.vc_coefficients(h, seed=5, contrast=4.0))
        g.set_vc_relax_shape(shape)
        g.setSolverParameters(sp, rp)
        g.set_bottom_params(imax=4)
        g.set_field(g.RHS, rhs)
        hist, _ = g.solve()
        runs.append((hist, g.get_field(g.PHI)))
        g.close()
    np.testing.assert_array_equal(runs[0][0], runs[1][0])
    np.testing.assert_array_equal(runs[0][1], runs[1][1])
