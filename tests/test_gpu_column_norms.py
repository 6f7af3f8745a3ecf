"""The column norms a solve reports (block partials and one finishing block a
system) for one, a few and many systems."""
import numpy as np
import pytest

import cassandra_amd.capi as capi
from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("systems", [1, 3, 17])
def test_column_norms_of_a_solve(ctx, systems):
    """The norms a PCG solve reports, from FP64 products of its solution (sums
    of 1e5 squares in another order: 1e-10)."""
    print(systems, flush=True)
    P = Patterns(ctx, N.FIT4)
    begin = np.cumsum([0] + [2000 + 700 * s for s in range(systems)])
    A = P.matrix_systems(ctx.random_play(41, int(begin[-1]), 20), begin)
    _, b = A.make_targets(42, 43)
    x, _, rel, _ = A.solve_systems(b, solver=capi.SOLVER_PCG, precision=capi.PREC_FP64, tol=0.0, max_iterations=3,
                                   check_every=3)
    norm = lambda y: A.spmtv(y).view(systems, P.cols).norm(dim=1)  # noqa: E731
    want = norm(b - A.spmv(x)) / norm(b)
    assert np.all(np.abs(rel - want.cpu().numpy()) <= 1e-10 * want.cpu().numpy())
