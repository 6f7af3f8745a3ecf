"""The differentiable evaluator's forward at every way its row loop can end:
slots below, at and above the steps of 4, 8, 12 and 20 entries, odd and even,
rows aligned to 8 bytes or not, entries outside the weights (which add
nothing).  The sum runs in slot order from zero (Pattern/Evaluator.cpp:48-54),
so it equals the oracle's product bit for bit."""
import numpy as np
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.evaluator import pattern_eval
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


def masks_of(k):
    """A pattern set of k slots, from patterns of 8, 4, 2 and 1 variations."""
    masks = []
    for order, pool in ((8, [N.B4, N.B5, N.test_a, N.B6, N.B4]), (4, [N.Q3]), (2, [N.test_vh]), (1, [N.test_vhdc])):
        for m in pool:
            if k >= order:
                masks.append(m)
                k -= order
    assert k == 0
    return masks


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 8, 9, 12, 13, 18, 19, 20, 21, 24, 28, 29, 32, 33, 40, 41])
def test_row_sums(ctx, oracle, k):
    print("slots", k, flush=True)
    masks = masks_of(k)
    P = Patterns(ctx, masks)
    assert P.k == k
    rows = 1021
    pos = oracle.random_play(900 + k, rows, 12, 40)
    idx = oracle.Group(masks).indices(pos).astype(np.int64)
    rng = np.random.default_rng(k)
    bad = rng.random(idx.shape) < 0.05
    given = np.where(bad, rng.choice([-1, P.cols, 2 ** 31 - 1], size=idx.shape), idx).astype(np.int32)
    for dtype in (torch.float32, torch.float64):
        w = torch.from_numpy(rng.standard_normal(P.cols)).to(dtype).cuda()
        # the entries that add nothing read a column of zero weight behind the others
        wz = np.concatenate([w.cpu().numpy(), np.zeros(1, w.cpu().numpy().dtype)])
        want = np.zeros(rows, wz.dtype)
        for s in range(k):
            want = want + wz[np.where(bad[:, s], P.cols, idx[:, s])]
        flat = torch.zeros(rows * k + 1, dtype=torch.int32, device="cuda")
        for shift in (0, 1):
            view = flat[shift:shift + rows * k].view(rows, k)
            view.copy_(torch.from_numpy(given))
            got = pattern_eval(w, view, P)
            assert np.array_equal(got.cpu().numpy(), want)
