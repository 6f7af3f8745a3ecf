"""The column sums over a window's partial slices (A^T y's second stage): one
slice a column up to several groups of sixteen, for each value type.  Integer y
makes every sum exact, so the products equal the oracle's
(Math/MatrixCSR.cpp:67-87), whatever the slices."""
import sys

import numpy as np
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


# one window (10,206 columns): a slice per 1,024 rows
@pytest.mark.parametrize("slices", [1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 31, 32, 33, 41])
def test_column_sums(ctx, oracle, slices):
    print("slices", slices, flush=True)
    sys.stdout.flush()
    rows = 1024 * slices - 7
    pos = oracle.random_play(300 + slices, rows, 12, 40)
    masks = [N.Q3]
    idx = oracle.Group(masks).indices(pos)
    A = Patterns(ctx, masks).matrix(torch.from_numpy(pos.view(np.int64)).cuda())
    y = np.random.default_rng(slices).integers(-64, 65, rows).astype(np.float64)
    want = oracle.spmtv(idx, y, A.cols)
    for dtype in (torch.float32, torch.float64):
        z = A.spmtv(torch.from_numpy(y).cuda().to(dtype)).cpu().numpy()
        assert np.array_equal(z.astype(np.float64), want)
    assert np.array_equal(A.jacobi().cpu().numpy(), oracle.jacobi(idx, A.cols), equal_nan=True)


# a batch: systems of one slice a column beside one of several
def test_batch_of_few_slices(ctx, oracle):
    print("batch of few slices", flush=True)
    rows = [400, 3000, 9000] + [400] * 21
    rb = np.concatenate([[0], np.cumsum(rows)])
    pos = oracle.random_play(401, int(rb[-1]), 12, 40)
    P = Patterns(ctx, N.FIT4)
    A = P.matrix_systems(torch.from_numpy(pos.view(np.int64)).cuda(), rb)
    y = np.random.default_rng(7).integers(-64, 65, A.rows).astype(np.float64)
    z = {d: A.spmtv(torch.from_numpy(y).cuda().to(d)).cpu().numpy() for d in (torch.float32, torch.float64)}
    g = oracle.Group(N.FIT4)
    for s in range(len(rows)):
        lo, hi = int(rb[s]), int(rb[s + 1])
        want = oracle.spmtv(g.indices(pos[lo:hi]), y[lo:hi], P.cols)
        for v in z.values():
            assert np.array_equal(v[s * P.cols:(s + 1) * P.cols].astype(np.float64), want)


# more windows than half the CUs (131 of 20,352 columns): two waves of tiles
@pytest.mark.parametrize("rows", [3, 5000, 40001])
def test_many_windows(ctx, oracle, rows):
    print("many windows", rows, flush=True)
    masks = [N.B6] * 5
    pos = oracle.random_play(600 + rows, rows, 12, 40)
    idx = oracle.Group(masks).indices(pos)
    A = Patterns(ctx, masks).matrix(torch.from_numpy(pos.view(np.int64)).cuda())
    y = np.random.default_rng(rows).integers(-64, 65, rows).astype(np.float64)
    want = oracle.spmtv(idx, y, A.cols)
    for dtype in (torch.float32, torch.float64):
        z = A.spmtv(torch.from_numpy(y).cuda().to(dtype)).cpu().numpy()
        assert np.array_equal(z.astype(np.float64), want)
