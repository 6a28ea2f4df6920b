"""Products of 1 to 16 rows, group 64, on the dense kernel: rows and columns at
the edges of its tiles (4, 8 and 16 rows; 32 columns), K of one group, of one
chunk and pass and past them, planes that are not 16-byte aligned (7 or 9
groups a row, odd row counts), corrections, codes, plane and output types and
D-ops, against the oracle (bar of tests/tolerances.py); batches of several
products against single ones."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests import test_gpu_affine as A
from tests.tolerances import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("m,n,k", [(1, 1, 64), (1, 33, 576), (2, 40, 448), (3, 96, 1024), (4, 31, 1088), (5, 64, 2112),
                                   (8, 100, 3136), (9, 17, 192), (16, 160, 2624)])
def test_dense_shapes(qmm, oracle, bits, layout, m, n, k):
    A.run_case(qmm, oracle, m=m, n=n, k=k, bits=bits, gs=64, layout=layout, seed=n + k + m)


@pytest.mark.parametrize("correction,signed,w_dt", [(0, False, H.BF16), (1, True, H.F16), (0, True, H.F16)])
@pytest.mark.parametrize("bits,m", [(4, 3), (4, 12), (8, 7)])
def test_dense_corrections(qmm, oracle, correction, signed, w_dt, bits, m):
    A.run_case(qmm, oracle, n=72, k=1216, m=m, bits=bits, gs=64, layout=0, correction=correction, signed=signed, w_dt=w_dt,
           seed=m)


# 8-bit products of five to eight rows (m, n, k), and whether the rule leaves them to qmv_mfma
W8_ROWS = [(5, 1536, 448, True), (6, 2048, 1024, True), (8, 8704, 2112, True), (7, 1536, 1088, False), (8, 8192, 2112, False)]


@pytest.mark.parametrize("m,n,k,mfma", W8_ROWS)
def test_w8_five_to_eight_rows(qmm, oracle, m, n, k, mfma):
    A.run_case(qmm, oracle, m=m, n=n, k=k, bits=8, gs=64, layout=1, seed=n + k + m)
    A.run_case(qmm, oracle, m=m, n=n, k=k, bits=8, gs=64, layout=1, correction=0, signed=True, w_dt=H.F16, accumulate=True,
               with_bias=True, seed=m)


@pytest.mark.parametrize("m", [1, 2])
def test_few_rows_in_one_launch(qmm, oracle, m):
    """A launch whose shorter products leave qmv_mfma's passes idle: all of them
    dense, the 4096-deep one (another kernel's when alone) included; and a
    product with unreadable planes beside readable ones, dragged and (past 160
    MB of others) not: each as the oracle has it."""
    rng = np.random.default_rng(m)
    kern = qmm.MatmulKernel(H.BF16, H.BF16, H.F32)
    for sizes in (((64, 1088), (48, 1088), (32, 4096)), ((33, 704), (64, 1024), (64, 4096)), ((33, 704), (81920, 4096))):
        args, cases = [], []
        for n, k in sizes:
            w = H.affine_weights(oracle, rng, min(n, 64), k, 4, 64, 0, 1, H.BF16)
            reps = -(-n // 64)  # a wide product repeats its rows
            x = H.activations(oracle, rng, m, k, H.BF16)
            codes, s, b = (H.to_dev(np.tile(w[key].reshape(min(n, 64), -1), (reps, 1)).ravel()) for key in ("codes", "scales", "corr"))
            d = torch.zeros(m * n, dtype=torch.float32, device="cuda")
            args.append(qmm.MatmulArguments(a=H.to_dev(x), m=m, n=n, k=k, d=d,
                                            b=qmm.QuantizedB(codes=codes, scales=s, correction_data=b,
                                                             params=qmm.QuantParams(0, n, k // 64))))
            cases.append((w, x, min(n, 64), k, n, d))
        kern.encode_many(args)
        torch.cuda.synchronize()
        for w, x, rows, k, n, d in cases:
            st, want = oracle.matmul(a=x, m=m, n=rows, k=k, codes=w["codes"], scales=w["scales"], correction_data=w["corr"],
                                     layout=0, bits=4, group_size=64, output_dt=H.F32, threads=8)
            assert st == 0
            mag = H.dequant_magnitude(oracle, w["codes"], w["scales"], w["corr"], rows, k, 4, 64, 0, 1, H.BF16, x, H.BF16, m)
            got = d.cpu().numpy().reshape(m, n)
            for r in (0, n - rows):
                check(got[:, r:r + rows].ravel(), want, mag=mag, label=f"m{m} n{n} k{k} at {r}")


@pytest.mark.parametrize("bits", [4, 8])
def test_dense_d_ops(qmm, oracle, bits):
    for m, dt in ((2, H.F32), (6, H.BF16), (11, H.F16)):
        A.run_case(qmm, oracle, m=m, n=45, k=832, bits=bits, ab_scale=0.75, accumulate=True, with_bias=True, soft_cap=4.0,
                   d_dt=dt, seed=m)


@pytest.mark.parametrize("bits,m", [(4, 1), (4, 6), (8, 8), (4, 16)])
def test_dense_batch_matches_single(qmm, oracle, bits, m):
    """Five products in one call, of different K and N, some of them another kernel's when alone."""
    rng = np.random.default_rng(bits + m)
    kern = qmm.MatmulKernel(H.BF16, H.BF16, H.BF16)
    args, outs = [], []
    for n, k in ((200, 704), (33, 704), (64, 2112), (512, 1024), (40, 128)):
        w = H.affine_weights(oracle, rng, n, k, bits, 64, 1, 1, H.BF16)
        x = H.to_dev(H.activations(oracle, rng, m, k, H.BF16))
        b = qmm.QuantizedB(codes=H.to_dev(w["codes"]), scales=H.to_dev(w["scales"]), params=qmm.QuantParams(1, n, k // 64),
                           mode=qmm.MODE_U4 if bits == 4 else qmm.MODE_U8, correction_data=H.to_dev(w["corr"]))
        for _ in range(2):
            outs.append(torch.zeros(m * n, dtype=torch.int16, device="cuda"))
            args.append(qmm.MatmulArguments(a=x, m=m, n=n, k=k, d=outs[-1], b=b))
    kern.encode_many(args[0::2])
    for a in args[1::2]:
        kern.encode_many([a])
    torch.cuda.synchronize()
    for a, b in zip(outs[0::2], outs[1::2]):
        got, want = (H.load(oracle, H.from_dev(t, np.uint16), H.BF16).astype(np.float64) for t in (a, b))
        # the same kernel gives the same bits; another one another order of the f32 sums (one bf16 ulp)
        assert np.all(np.abs(got - want) <= 2.0 ** -7 * np.abs(want) + 1e-3 * np.abs(want).max())


@pytest.mark.parametrize("bits,m,bar", [(4, 16, 1.62e-7), (8, 8, 1.48e-7), (8, 16, 1.48e-7)])
def test_dense_sums_against_64_bits(qmm, bits, m, bar):
    """f32 sums over 12288 values, 24 groups a wave. One chain that rounds twice a
    group at the running sum's size measured 1.74e-7 (4-bit) and 1.60e-7 (8-bit);
    two chains, or one rounding a group, halve the error variance that grows with
    K: 1.50e-7 and 1.37e-7. The bars lie between."""
    g = torch.Generator(device="cuda").manual_seed(bits)
    n, k, levels = 1000, 12288, (1 << bits) - 1
    w = torch.randn(n, k // 64, 64, generator=g, device="cuda") * 0.02
    lo, hi = w.amin(dim=2), w.amax(dim=2)
    s, b = ((hi - lo) / float(levels)).to(torch.bfloat16), lo.to(torch.bfloat16)
    q = torch.round((w - b.float().unsqueeze(2)) / s.float().unsqueeze(2)).clamp_(0, levels).to(torch.uint8).view(n, k)
    codes = (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous() if bits == 4 else q.contiguous()
    x = torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16)
    d = torch.zeros(m, n, device="cuda")
    qmm.MatmulKernel(H.BF16, H.BF16, H.F32).encode(qmm.MatmulArguments(
        a=x, m=m, n=n, k=k, d=d, b=qmm.QuantizedB(codes=codes, scales=s, correction_data=b, params=qmm.QuantParams(0, n, k // 64),
                                                  mode=qmm.MODE_U4 if bits == 4 else qmm.MODE_U8)))
    torch.cuda.synchronize()
    f64 = (q.double().view(n, -1, 64) * s.double().unsqueeze(2) + b.double().unsqueeze(2)).view(n, k)
    want = x.double() @ f64.t().contiguous()
    assert ((d.double() - want).norm() / want.norm()).item() < bar
