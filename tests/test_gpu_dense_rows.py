"""bf16 products by blocks of rows: activation rows at the edges of its blocks
(1, 4, 8), weight rows that are no multiple of four on both sides of the rule
that takes four a workgroup, K below and past a step of 2048, against the
oracle; a row's bits do not depend on the number of rows."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests import test_gpu_dense as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 3, 8), (2, 130, 2056), (4, 7, 4096), (5, 33, 504), (8, 2051, 512), (9, 129, 2048),
                                   (130, 127, 1024)])
def test_dense_row_blocks(qmm, oracle, m, n, k):
    D.run(qmm, oracle, m, n, k, seed=m + n)


def test_dense_rows_do_not_depend_on_the_batch(qmm, oracle):
    rng = np.random.default_rng(5)
    n, k, m = 126, 2056, 300
    w = H.to_dev(H.store(oracle, rng.normal(0, 0.05, n * k).astype(np.float32), H.BF16))
    x = H.to_dev(H.store(oracle, rng.normal(0, 1, m * k).astype(np.float32), H.BF16))
    kern = qmm.MatmulKernel(H.BF16, H.BF16, H.F32)

    def product(rows):
        d = torch.zeros(rows * n, dtype=torch.float32, device="cuda")
        kern.encode(qmm.MatmulArguments(a=x, b=qmm.FullPrecisionB(values=w), d=d, m=rows, n=n, k=k))
        return d

    whole = product(m)
    for rows in (1, 3, 4, 8, 60):
        assert torch.equal(product(rows), whole[:rows * n])
