"""The resident evaluator's kernels against the oracle's sum in slot order, bit
for bit: batches around the 64 positions of a small block, around the size from
which the weights are staged in LDS and around one pass of the chip there;
pattern sets whose weights all fit the LDS, partly, or not at all, and one with
more index tiles than a block has waves; host batches on both sides of the
pinned limit."""
import numpy as np
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu

SETS = {"small": N.test_mix + [N.L1], "part": N.cassandra, "none": [N.B5, N.B6], "tiles": N.FIT12 + N.edax}


@pytest.mark.parametrize("name", list(SETS))
def test_sizes(ctx, oracle, name):
    masks = SETS[name]
    P, g = Patterns(ctx, masks), oracle.Group(masks)
    w = np.random.default_rng(7).normal(size=P.cols).astype(np.float32)
    E = P.evaluator(torch.from_numpy(w).cuda())
    pos = oracle.random_play(17, 600_001, 4, 56)
    want = oracle.spmv(g.indices(pos), w)
    d = torch.from_numpy(pos.view(np.int64)).cuda()
    for n in (1, 63, 64, 65, 1000, 131_071, 131_072, 131_073, 262_145, 524_289, 600_001):
        print(name, n, flush=True)
        assert np.array_equal(E(d[:n].contiguous()).cpu().numpy(), want[:n])
    for n in (1, 255, 257, 16_384, 16_385, 300):
        print(name, "host", n, flush=True)
        assert np.array_equal(E.eval_host(pos[:n]), want[:n])
