"""Slot-major extraction of many rows (four rows a lane): sizes around a wave's
256 rows and around the line from which it runs, written at aligned and
unaligned places, and the stored matrix's 2-byte form of the same indices
(Pattern/Indexer.cpp:413-422 forms a row)."""
import ctypes as C

import numpy as np
import pytest
import torch

import cassandra_amd.capi as capi
from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [524287, 524288, 524289, 524290, 524544, 524545, 600001, 600127])
def test_slot_major_equals_rows(ctx, oracle, rows):
    print("slot-major extraction", rows, flush=True)
    masks = [N.Q3, N.B4, N.test_vhdc]
    P = Patterns(ctx, masks)
    pos = ctx.random_play(rows, rows, 12, 40)
    want = P.extract(pos)
    head = oracle.Group(masks).indices(pos[-300:].cpu().numpy().view(np.uint64))
    assert np.array_equal(want[-300:].cpu().numpy().astype(np.int64), head.astype(np.int64))
    for shift in (0, 1, 3):
        out = torch.full((P.k * rows + 8,), -7, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        capi.call("cad_index_extract", P.h, C.c_void_p(pos.data_ptr()), rows,
                  C.c_void_p(out[shift:].data_ptr()), capi.LAYOUT_SLOT_MAJOR)
        ctx.synchronize()
        assert torch.equal(out[shift:shift + P.k * rows].view(P.k, rows).t(), want)
        assert bool((out[:shift] == -7).all()) and bool((out[shift + P.k * rows:] == -7).all())
    assert np.array_equal(P.matrix(pos).download()[-300:], head)
