"""cad_matrix_kernel_times reports the parts that an FP32 product launches: a
stored matrix's A^T y has a max |y| pass over its row blocks, a matrix-free one
(FP64 windows) has none; and it leaves the matrix's products as they were."""
import pytest
import torch

from cassandra_amd import names as N
from cassandra_amd.fit import Patterns

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("free", [False, True])
def test_parts_of_a_product(ctx, free):
    print("kernel times", "matrix-free" if free else "stored", flush=True)
    P = Patterns(ctx, N.FIT4)
    pos = ctx.random_play(5, 20001, 20)
    A = P.matrix_free(pos) if free else P.matrix(pos)
    y = torch.randint(-64, 65, (A.rows,), device="cuda").float()
    z = A.spmtv(y)
    t = A.kernel_times(5)
    assert all(t[k] > 0 for k in ("gather", "scatter_tiles", "scatter_reduce", "jacobi_part"))
    assert (t["absmax"] == 0) == free
    assert torch.equal(A.spmtv(y), z)
