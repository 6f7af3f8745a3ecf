"""FP32 A^T y of a matrix-free matrix: every term (an FP32 value) is added to
FP64 windows, so a column's error is the FP32 rounding of its own sums
(Math/MatrixCSR.cpp:67-87 forms the same sums), whatever the range of y: the
largest |y| costs no other column a bit.

The bound: a window's partial slices and the result are each rounded to FP32
once (2^-24 of the slices' absolute sum and of the result), the FP64 sums add
less than 2^-40: 2e-7 of |A|^T |y| a column."""
import sys

import numpy as np
import pytest
import torch

import cassandra_amd.capi as capi
from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def values(kind, n, rng):
    y = rng.standard_normal(n).astype(np.float32)
    if kind == "wide":  # 60 binary orders, every row its own
        y *= np.exp2(rng.uniform(-50.0, 10.0, n)).astype(np.float32)
    elif kind == "spike":  # one row far above the rest
        y[n // 3] = 1e30
    elif kind == "small":
        y *= np.float32(1e-30)
    elif kind in ("nan", "inf"):
        y[n // 3] = float(kind)
    return y


# 64 and 1,024 rows and one beside; packed groups of 32 slots (FIT12, edax)
@pytest.mark.parametrize("masks", [N.FIT12, N.edax, N.test_mix])
@pytest.mark.parametrize("rows", [1, 63, 65, 1025, 50001])
@pytest.mark.parametrize("kind", ["normal", "wide", "spike", "small", "nan", "inf"])
def test_transposed_product_keeps_fp32(ctx, oracle, masks, rows, kind):
    say("matrix-free FP32 A^T y", len(masks), rows, kind)
    pos = oracle.random_play(7000 + rows, rows, 15, 45)
    idx = oracle.Group(masks).indices(pos)
    F = Patterns(ctx, masks).matrix_free(torch.from_numpy(pos.view(np.int64)).cuda())
    y = values(kind, rows, np.random.default_rng(rows))
    z = F.spmtv(torch.from_numpy(y).cuda()).cpu().numpy().astype(np.float64)
    bad = ~np.isfinite(y)
    hit = np.zeros(F.cols, bool)
    hit[np.unique(idx[bad])] = True
    y64 = np.where(bad, 0.0, y.astype(np.float64))
    exact = oracle.spmtv(idx, y64, F.cols)
    bound = 2e-7 * oracle.spmtv(idx, np.abs(y64), F.cols) + 2.0 ** -149  # (a subnormal's own rounding)
    assert np.all(~np.isfinite(z[hit]))
    assert np.all(np.abs(z[~hit] - exact[~hit]) <= bound[~hit])


def test_pcg_matches_stored(ctx, oracle):
    """Two FP32 PCG iterations on a matrix-free matrix.  A product errs by about
    2e-7 of its absolute sums, ten times that relative to the sums themselves;
    the second residual is a difference that loses another digit, and the step
    along it a few times that: 1e-4 of the predictions."""
    say("matrix-free FP32 PCG")
    pos = oracle.random_play(81, 20000, 15, 45)
    idx = oracle.Group(N.FIT12).indices(pos)
    P = Patterns(ctx, N.FIT12)
    d = torch.from_numpy(pos.view(np.int64)).cuda()
    S, F = P.matrix(d), P.matrix_free(d)
    _, b = S.make_targets(2006, 3006)
    opts = dict(solver=capi.SOLVER_PCG, tol=0.0, max_iterations=2, check_every=2)
    want = oracle.spmv(idx, S.solve(b, precision=capi.PREC_FP64, **opts)[0].cpu().numpy())
    for A in (S, F):
        got = oracle.spmv(idx, A.solve(b, precision=capi.PREC_FP32, **opts)[0].cpu().numpy())
        assert np.linalg.norm(got - want) <= 1e-4 * np.linalg.norm(want)
