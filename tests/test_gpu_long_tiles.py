"""A x over long tiles (more than one run of rows a thread and tile) against the
oracle, bit for bit: the row counts at which the plan takes one, two and three
runs, with ragged ends, and batches whose small systems hold fewer rows than a
run."""
import numpy as np
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


def check(A, idx, oracle, dtype, seed=5):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(A.cols, dtype=dtype, device="cuda", generator=gen)
    got = A.spmv(x).cpu().numpy()
    assert np.array_equal(got, oracle.spmv(idx, x.cpu().numpy()))


@pytest.mark.parametrize("rows,dtype", [(530_003, torch.float64), (1_200_003, torch.float64),
                                        (2_300_001, torch.float32), (4_300_007, torch.float32)])
def test_single_system(ctx, oracle, rows, dtype):
    print(rows, dtype, flush=True)
    pos = ctx.random_play(31, rows, 22)
    idx = oracle.Group(N.FIT4).indices(pos.cpu().numpy().view(np.uint64))
    check(Patterns(ctx, N.FIT4).matrix(pos), idx, oracle, dtype)


@pytest.mark.parametrize("dtype,sizes", [(torch.float64, [1, 3001, 400_001, 700_003]),
                                         (torch.float32, [5, 2_400_001, 30_007])])
def test_batch(ctx, oracle, dtype, sizes):
    print(sizes, dtype, flush=True)
    begin = np.concatenate([[0], np.cumsum(sizes)])
    pos = ctx.random_play(32, int(begin[-1]), 22)
    P = Patterns(ctx, N.FIT4)
    idx = oracle.Group(N.FIT4).indices(pos.cpu().numpy().view(np.uint64))
    for s in range(len(sizes)):
        idx[begin[s]:begin[s + 1]] += np.uint32(s * P.cols)
    check(P.matrix_systems(pos, begin), idx, oracle, dtype)
