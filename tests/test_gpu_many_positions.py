"""More positions than one launch of a thread a slot group and row can hold: the
evaluator's block kernel, which scores every set whose patterns are all too wide
for the LDS, over 2^28 positions and a few (Pattern/Evaluator.cpp:48-54)."""
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


def test_scores_of_2_28_positions(ctx):
    print("scores of 2^28 positions", flush=True)
    # 16 index tiles, 16 waves a block
    P = Patterns(ctx, [N.B5] * 8)
    w = torch.randn(P.cols, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    E = P.evaluator(w)
    base = ctx.random_play(17, 1 << 20, 12, 40)
    want = E(base)
    n = (1 << 28) + 65
    pos = torch.empty((n, 2), dtype=torch.int64, device="cuda")
    for a in range(0, n, 1 << 20):
        pos[a:a + (1 << 20)] = base[:min(1 << 20, n - a)]
    got = E(pos)
    assert torch.equal(got[:1 << 28].view(256, 1 << 20), want.expand(256, 1 << 20))
    assert torch.equal(got[1 << 28:], want[:65])
