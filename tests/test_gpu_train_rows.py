"""The fused training step over row lengths of one chunk of slots, its edges and
several, and minibatches with ragged waves, against the same epochs through
torch: the minibatch losses depend on every entry of the step before (float
means of at most 300 terms: 2e-5)."""
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.evaluator import huber_fit, huber_fit_fused
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu

# k = 1 (a fully symmetric mask), 18, 32, 34, 54, 100
SETS = {1: [N.test_vhdc], 18: N.FIT4, 32: N.FIT8[:3] + N.FIT8[4:], 34: N.FIT8, 54: N.FIT12, 100: N.FIT12 + N.edax}


@pytest.mark.parametrize("k", list(SETS))
@pytest.mark.parametrize("rows,batch", [(1, 1), (65, 64), (300, 129)])
def test_losses(ctx, k, rows, batch):
    print(k, rows, batch, flush=True)
    P = Patterns(ctx, SETS[k])
    assert P.k == k
    pos = ctx.random_play(3, rows, 20)
    idx = P.extract(pos)
    target = P.matrix(pos).make_targets(4, 5)[1].float()
    a = huber_fit(P, idx, target, epochs=3, batch=batch, seed=6)[1]
    b = huber_fit_fused(P, idx, target, epochs=3, batch=batch, seed=6)[1]
    assert a == pytest.approx(b, rel=2e-5, abs=1e-6)
