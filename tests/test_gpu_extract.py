"""Index extraction on the device against the host's index programs: the index
tiles (matrix products of the digits) of every kind of pattern, and the two
layouts' store paths."""
import numpy as np
import pytest
import torch

import cassandra_amd.capi as capi
from cassandra_amd import names as N

pytestmark = pytest.mark.gpu


def _mask(squares):
    return sum(1 << (x + 8 * y) for x, y in squares)


# Patterns whose lists need more than five or ten digits: the largest
# symmetric ones (16 squares: a half-pattern number reaches 3^8 and a pair's
# index 21.5 million, past 24 bits), seven squares a half with a diagonal list,
# and 11 to 16 squares without symmetry.
_HALF = [(1, 0), (2, 0), (3, 0), (4, 0), (2, 1), (3, 1), (4, 1), (3, 2)]
WIDE = {
    "diagonal_16": _mask(_HALF + [(y, x) for x, y in _HALF]),
    "diagonal_7_2": _mask(_HALF[:7] + [(y, x) for x, y in _HALF[:7]] + [(0, 0), (1, 1)]),
    "diagonal_6_1": _mask(_HALF[:6] + [(y, x) for x, y in _HALF[:6]] + [(5, 5)]),
    "vertical_16": 0xFFFF,
    "vertical_12": 0x3CFF,
    "none_11": 0x00000000000F3F01,
    "none_16": 0x0000000080FF7E01,
}


def check(ctx, masks, n, seed=77):
    from cassandra_amd.fit import Patterns

    P = Patterns(ctx, masks)
    pos = ctx.random_play(seed, n, 0, 40)
    want = P.indices_host(pos.cpu().numpy().view(np.uint64))
    got = P.extract(pos).cpu().numpy().view(np.uint32)
    assert np.array_equal(got, want), "row-major"
    got = P.extract(pos, capi.LAYOUT_SLOT_MAJOR).cpu().numpy().view(np.uint32)
    assert np.array_equal(got.T, want), "slot-major"
    return P, pos, want


@pytest.mark.parametrize("name", sorted(WIDE))
def test_long_lists(ctx, name):
    print(name, flush=True)
    check(ctx, [WIDE[name]], 1037)


# one store run per wave (k = 18), several chunks of slots a row (k = 88), one
# and two slots per pattern; rows below, at and past a wave's 64
@pytest.mark.parametrize("n", [1, 63, 64, 65, 1027])
@pytest.mark.parametrize("masks", [N.FIT4, N.FIT12 + N.FIT8, N.test_mix, [N.D8], [N.test_vhdc]],
                         ids=["k18", "k88", "mix", "k2", "k1"])
def test_layouts(ctx, masks, n):
    print(len(masks), n, flush=True)
    check(ctx, masks, n)


# enough rows for four a lane: aligned runs (a matrix's slots, u16 and u32
# entries) and slots that start at odd rows (the caller's slot-major array),
# with a last wave that is partly past the end
@pytest.mark.parametrize("masks", [N.FIT4, [N.B6, N.D8]], ids=["u16", "u32"])
def test_many_rows(ctx, masks):
    n = 64 * 4 * 8 * 256 + 77
    print(len(masks), n, flush=True)
    P, pos, want = check(ctx, masks, n)
    A = P.matrix(pos)
    assert np.array_equal(A.download(), want)
    y = A.spmtv(torch.ones(n, dtype=torch.float64, device="cuda"))
    assert np.array_equal(y.cpu().numpy(), np.bincount(want.ravel(), minlength=A.cols))
