"""The differentiable evaluator's backward at the edges of its row steps (1,024
rows of a block and one beside, the second row of a thread there or not) and for
groups of one to eight slots.  Integer g makes the sums exact: grad_w equals the
oracle's A^T g (Math/MatrixCSR.cpp:67-87)."""
import numpy as np
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.evaluator import pattern_eval
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu

SETS = {
    "one slot": [N.test_vhdc],
    "two slots": [N.test_vh],
    "four slots": [N.Q3],
    "four slots, windows": [N.L02X],
    "eight slots, windows": [N.B5],
    "packed": [N.D4, N.D5, N.test_vh, N.Q3],
    "FIT4": N.FIT4,
}


@pytest.mark.parametrize("name", sorted(SETS))
@pytest.mark.parametrize("rows", [1, 1023, 1024, 1025, 2047, 2048, 2049, 3073, 65537])
def test_gradient(ctx, oracle, name, rows):
    print("backward", name, rows, flush=True)
    P = Patterns(ctx, SETS[name])
    pos = oracle.random_play(500 + rows % 97, rows, 12, 40)
    idx = oracle.Group(SETS[name]).indices(pos)
    g = np.random.default_rng(rows).integers(-64, 65, rows).astype(np.float64)
    want = oracle.spmtv(idx, g, P.cols)
    di = torch.from_numpy(idx.astype(np.int32)).cuda()
    for dtype in (torch.float32, torch.float64):
        w = torch.zeros(P.cols, dtype=dtype, device="cuda", requires_grad=True)
        (grad,) = torch.autograd.grad(pattern_eval(w, di, P), w, torch.from_numpy(g).cuda().to(dtype))
        assert np.array_equal(grad.cpu().numpy().astype(np.float64), want)
