"""qmv_small_m (4-bit, group 64, 9 to 16 rows, K % 1024 == 0, launches with many
passes for each resident workgroup): each case runs beside a product that makes
its launch long (helpers.long_launch; that this is enough for the rule is
asserted on the CPU, test_dispatch_rules.py). One tile, a pair with a shifted
second tile, ragged N; runs of one, two and three pairs (K of 12288, 4096 and
1024 values beside it); corrections, codes, planes and D-ops; batches."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests import test_gpu_affine as A

pytestmark = pytest.mark.gpu

SHAPES = [(16, 1024), (17, 2048), (40, 4096), (1000, 2048), (96, 12288), (9000, 1024)]
ROWS = [9, 12, 16]


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize("layout", [0, 1])
def test_shapes(qmm, oracle, n, k, m, layout):
    A.run_case(qmm, oracle, m=m, n=n, k=k, layout=layout, seed=n + k + 3 * m + layout, long_launch=True)


@pytest.mark.parametrize("correction,signed,w_dt", [(0, False, H.BF16), (1, True, H.BF16), (1, False, H.F16), (0, True, H.F16)])
def test_variants(qmm, oracle, correction, signed, w_dt):
    A.run_case(qmm, oracle, m=11, n=72, k=2048, correction=correction, signed=signed, w_dt=w_dt, seed=17 + correction,
               long_launch=True)


@pytest.mark.parametrize("d_dt", [H.F32, H.BF16, H.F16])
def test_d_ops(qmm, oracle, d_dt):
    A.run_case(qmm, oracle, m=13, n=40, k=1024, ab_scale=0.75, accumulate=True, with_bias=True, soft_cap=30.0, d_dt=d_dt,
               seed=5, long_launch=True)


def test_run_length_keeps_bits(qmm, oracle):
    """Products of three depths in one long launch and each beside the long one alone: the same bits, whatever the run."""
    rng = np.random.default_rng(37)
    kern = qmm.MatmulKernel(H.BF16, H.BF16, H.BF16)
    args, outs = [], []
    for n, k in ((512, 12288), (1024, 4096), (2048, 1024)):
        w = H.affine_weights(oracle, rng, n, k, 4, 64, layout=1)
        x = H.to_dev(H.activations(oracle, rng, 10, k))
        b = qmm.QuantizedB(codes=H.to_dev(w["codes"]), scales=H.to_dev(w["scales"]), params=qmm.QuantParams(1, n, k // 64),
                           correction_data=H.to_dev(w["corr"]))
        for _ in range(2):
            outs.append(torch.zeros(10 * n, dtype=torch.int16, device="cuda"))
            args.append(qmm.MatmulArguments(a=x, m=10, n=n, k=k, d=outs[-1], b=b))
    kern.encode_many(args[0::2] + [H.long_launch(qmm, 10)])
    for a in args[1::2]:
        kern.encode_many([a, H.long_launch(qmm, 10)])
    torch.cuda.synchronize()
    for a, b in zip(outs[0::2], outs[1::2]):
        assert torch.equal(a, b)
