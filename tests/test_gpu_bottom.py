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
    ((29, 31, 30), ([15], [16], [14]), (0.3, 1.1), WALLS),             # 13950 slots: one colour, two stages
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
