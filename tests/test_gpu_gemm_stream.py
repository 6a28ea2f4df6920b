"""Prompt products of 17 to 128 rows, group 64, on the weight-streaming kernel:
rows at the edges of its row blocks (32, 48, 64; one and two blocks), ragged
columns at both widths (32 and 64 columns a workgroup), K of one group, of a
pass less one group and past several passes, both plane layouts, corrections,
codes, plane and output types and D-ops, against the oracle; the weights bit for
bit; batches against single products."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests import test_gpu_affine as A
from tests import test_gpu_exact_dequant as E
from tests import test_gpu_range as R
from tests.tolerances import check

pytestmark = pytest.mark.gpu


EXACT = [(17, 1, 64), (32, 33, 192), (33, 40, 320), (48, 97, 576), (49, 31, 1088), (64, 65, 2112), (65, 100, 832), (96, 17, 256),
         (97, 70, 1216), (128, 33, 512)]
# m, n, k, f16 planes and results; 64 columns a workgroup (else 32)
SUMS = [(20, 3000, 448, False, False), (40, 25000, 320, True, True), (64, 25000, 192, False, True), (100, 600, 3520, True, False),
        (128, 600, 4416, False, False), (24, 25000, 320, False, True), (60, 10000, 1088, True, True), (80, 5000, 832, False, True),
        (128, 8100, 576, False, True)]


@pytest.mark.parametrize("bits,layout", [(4, 0), (4, 1), (8, 0), (8, 1)])
@pytest.mark.parametrize("m,n,k", EXACT)
def test_stream_weights_exact(qmm, oracle, bits, layout, m, n, k):
    E._gemm_exact(qmm, oracle, n=n, k=k, bits=bits, layout=layout, seed=m + n + k, m=m, label="qgemm_stream")


@pytest.mark.parametrize("correction,signed", [(0, False), (1, True), (0, True)])
@pytest.mark.parametrize("bits,m", [(4, 30), (8, 50)])
def test_stream_corrections_exact(qmm, oracle, correction, signed, bits, m):
    E._gemm_exact(qmm, oracle, n=72, k=1216, bits=bits, correction=correction, signed=signed, seed=m, m=m, label="qgemm_stream")


@pytest.mark.parametrize("m,n,k,f16,wide", SUMS)
def test_stream_sums(qmm, oracle, m, n, k, f16, wide):
    """Both column widths against the f64 product of the bf16-effective weights, with the D-ops; f16 planes and results at two sizes."""
    A._short_prompt_case(qmm, oracle, m, n, k, seed=m + n, ab_scale=0.75, accumulate=True, with_bias=True, soft_cap=30.0,
                   w_dt=H.F16 if f16 else H.BF16, d_dt=H.BF16 if f16 else H.F32)


@pytest.mark.parametrize("bits", [4, 8])
def test_stream_batch_matches_single(qmm, oracle, bits):
    """Products of up to 64 rows, of different rows, K and N, in one call and alone: the same bits."""
    rng = np.random.default_rng(bits)
    kern = qmm.MatmulKernel(H.BF16, H.BF16, H.F32)
    args, outs = [], []
    for m, n, k in ((17, 200, 704), (48, 33, 704), (64, 13000, 128), (40, 13000, 192), (64, 40, 4416)):
        w = H.affine_weights(oracle, rng, n, k, bits, 64, 1, 1, H.BF16)
        x = H.to_dev(H.activations(oracle, rng, m, k, H.BF16))
        b = qmm.QuantizedB(codes=H.to_dev(w["codes"]), scales=H.to_dev(w["scales"]), params=qmm.QuantParams(1, n, k // 64),
                           mode=qmm.MODE_U4 if bits == 4 else qmm.MODE_U8, correction_data=H.to_dev(w["corr"]))
        for _ in range(2):
            outs.append(torch.zeros(m * n, dtype=torch.float32, device="cuda"))
            args.append(qmm.MatmulArguments(a=x, m=m, n=n, k=k, d=outs[-1], b=b))
    kern.encode_many(args[0::2])
    for a in args[1::2]:
        kern.encode(a)
    torch.cuda.synchronize()
    for a, b in zip(outs[0::2], outs[1::2]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,k,m", [(262100, 8192, 17), (40, 4194304 + 64, 32)])
def test_products_past_the_gemm_keep_f32_weights(qmm, n, k, m):
    """8-bit products that the GEMM's 32-bit offsets refuse (the last 128 rows
    below 2 GiB of codes; K past its activation rows) run on the kernels that
    keep the dequantized weights in f32, whatever their row count: bf16 weights
    would be 1.6e-3 off the 64-bit product, f32 ones and sums are below 1e-5."""
    g = torch.Generator(device="cuda").manual_seed(n)
    codes = torch.randint(0, 256, (n, k), generator=g, device="cuda", dtype=torch.uint8)
    s = (0.002 + 0.002 * torch.rand(n, k // 64, generator=g, device="cuda")).to(torch.bfloat16)
    b = (-128.0 * s.float() + 0.02 * torch.rand(n, k // 64, generator=g, device="cuda")).to(torch.bfloat16)
    x = torch.randn(m, k, generator=g, device="cuda").to(torch.bfloat16)
    d = torch.zeros(m, n, device="cuda")
    weights = qmm.QuantizedB(codes=codes, scales=s, correction_data=b, mode=qmm.MODE_U8,
                             params=qmm.QuantParams(qmm.OUTPUT_GROUP, n, k // 64))
    args = qmm.MatmulArguments(a=x, b=weights, d=d, m=m, n=n, k=k)
    kern = qmm.MatmulKernel(H.BF16, H.BF16, H.F32)
    for call in (lambda: kern.encode(args), lambda: kern.encode_many([args])):
        d.zero_()
        call()
        torch.cuda.synchronize()
        for r in (0, n - min(n, 64)):
            rows = slice(r, min(r + 64, n))
            w = codes[rows].double().view(-1, k // 64, 64) * s[rows].double().unsqueeze(2) + b[rows].double().unsqueeze(2)
            want = x.double() @ w.view(-1, k).t().contiguous()
            assert ((d[:, rows].double() - want).norm() / want.norm()).item() < 1e-5


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k", [(20, 48, 1088), (100, 96, 832)])
def test_stream_activation_range(qmm, oracle, bits, m, n, k):
    """Activations of 2^-100 to 2^70, groups of mixed magnitudes and bf16 subnormals, against the f64 product."""
    rng = np.random.default_rng(m + bits)
    w = H.affine_weights(oracle, rng, n, k, bits, 64, 1, 1, H.BF16)
    x = H.store(oracle, R.wide_x(rng, m, k), H.BF16)
    got = _product(qmm, w, x, m, n, k, bits)
    want, mag = A.bf16_effective_reference(oracle, w, x, m, n, k, bits, 64, 1, 1, H.BF16, False)
    check(got.ravel(), want.ravel(), mag=mag.ravel(), label=f"range m{m} b{bits}")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m", [20, 100])
def test_stream_non_finite_activations(qmm, oracle, bits, m):
    """A row with an infinity or a NaN is not finite where its f64 product with
    the same bf16 weights is not, with that sign; the others keep their bits."""
    rng = np.random.default_rng(m + bits)
    n, k = 80, 832
    w = H.affine_weights(oracle, rng, n, k, bits, 64, 1, 1, H.BF16)
    xf = rng.normal(0, 1, (m, k)).astype(np.float32)
    plain = _product(qmm, w, H.store(oracle, xf.ravel(), H.BF16), m, n, k, bits)
    xf[2, 5], xf[m - 1, k - 3], xf[7, 100] = np.inf, -np.inf, np.nan
    x = H.store(oracle, xf.ravel(), H.BF16)
    got = _product(qmm, w, x, m, n, k, bits)
    with np.errstate(invalid="ignore"):
        want, _ = A.bf16_effective_reference(oracle, w, x, m, n, k, bits, 64, 1, 1, H.BF16, False)
    bad = [2, 7, m - 1]
    assert np.array_equal(np.isnan(got[bad]), np.isnan(want[bad]))
    inf = np.isinf(want[bad])
    assert inf.any() and np.array_equal(np.sign(got[bad][inf]), np.sign(want[bad][inf])) and np.isinf(got[bad][inf]).all()
    rest = np.setdiff1d(np.arange(m), bad)
    assert np.array_equal(got[rest].view(np.uint32), plain[rest].view(np.uint32))


def _product(qmm, w, x, m, n, k, bits):
    d = torch.zeros(m * n, dtype=torch.float32, device="cuda")
    qmm.MatmulKernel(H.BF16, H.BF16, H.F32).encode(qmm.MatmulArguments(a=H.to_dev(x), m=m, n=n, k=k, d=d, b=qmm.QuantizedB(
        codes=H.to_dev(w["codes"]), scales=H.to_dev(w["scales"]), correction_data=H.to_dev(w["corr"]),
        params=qmm.QuantParams(1, n, k // 64), mode=qmm.MODE_U4 if bits == 4 else qmm.MODE_U8)))
    torch.cuda.synchronize()
    return d.cpu().numpy().reshape(m, n)
