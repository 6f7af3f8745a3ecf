"""Repeated FP32 PCG solves of one batch on the same matrix: launched directly at
first, from a captured graph once there were enough to pay for it.  The FP32
products and the sums of the recurrence are order-independent or fixed in order
(Math/Solver.h:100-155 is the iteration), so every solve gives the same bits,
also when the right side changes in between."""
import numpy as np
import pytest
import torch

import cassandra_amd.capi as capi
from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [3000, 30000])
def test_one_batch_solves_agree(ctx, rows):
    print("repeated solves", rows, flush=True)
    A = Patterns(ctx, N.FIT4).matrix(ctx.random_play(31, rows, 20))
    b1, b2 = A.make_targets(41, 51)[1], A.make_targets(42, 52)[1]
    opts = dict(solver=capi.SOLVER_PCG, precision=capi.PREC_FP32, tol=0.0, max_iterations=40, check_every=40)
    first = [A.solve(b, **opts)[0] for b in (b1, b2)]
    for i in range(20):
        b, want = ((b1, first[0]), (b2, first[1]))[i % 2]
        x, rep = A.solve(b, **opts)
        assert rep["iterations"] == 40
        assert torch.equal(x, want)
    # another batch length after the graph exists, and a run of several batches
    y = [A.solve(b1, **dict(opts, max_iterations=20, check_every=c))[0] for c in (20, 10, 5)]
    assert torch.equal(y[0], y[1]) and torch.equal(y[0], y[2])
    assert np.isfinite(y[0].cpu().numpy()).all()
