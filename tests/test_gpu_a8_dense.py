"""Int8-activation products on the weight-streaming kernel: every workgroup shape
its rule can choose, over several passes and an odd last group (SHAPES; which
shape a size gets is asserted on the CPU, test_dispatch_rules.py), both sides of
the rule that leaves one or two rows of few columns to a wave a row (ROWS), edges
of its tiles (rows, 32 to 256 columns) and passes, planes of any alignment, both
code layouts, activation groups of 64 and 128, corrections, codes and D-ops,
against the oracle (bar of tests/tolerances.py)."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests.tolerances import check

pytestmark = pytest.mark.gpu


def _run(Q, O, m, n, k, bits, ag, grouped, layout, correction=1, signed=False, w_dt=H.BF16, d_dt=H.F32, d_ops=False):
    rng = np.random.default_rng(m + n + k + bits)
    w = H.affine_weights(O, rng, n, k, bits, 64, layout, correction, w_dt)
    q = rng.integers(-127, 128, (m, k)).astype(np.int8)
    sc = rng.uniform(0.001, 0.1, (m, k // ag)).astype(np.float32)
    prior = H.store(O, rng.normal(0, 1, m * n).astype(np.float32), d_dt) if d_ops else None
    bias = H.store(O, rng.normal(0, 0.5, n).astype(np.float32), w_dt) if d_ops else None
    st, want = O.matmul(a=np.zeros(m * k, np.uint16), m=m, n=n, k=k, codes=w["codes"], scales=w["scales"], correction=correction,
                        correction_data=w["corr"], layout=layout, row_count=n, group_count=k // 64, bits=bits,
                        group_size=64, signed_codes=signed, d=prior, ab_scale=0.5 if d_ops else 1.0, accumulate=d_ops,
                        bias=bias, weights_dt=w_dt, input_dt=H.BF16, output_dt=d_dt, threads=8, a_codes=q.ravel(),
                        a_scales=sc.ravel(), a_scale_group_size=ag, a_grouped_by_nibble=bool(grouped))
    assert st == 0
    d = H.to_dev(prior) if d_ops else torch.zeros(m * n, dtype=torch.float32 if d_dt == H.F32 else torch.int16, device="cuda")
    a = Q.Int8SymmetricA(values=H.to_dev(q), scales=H.to_dev(sc), scale_group_size=ag,
                         code_layout=Q.GROUPED_BY_NIBBLE if grouped else Q.SEQUENTIAL)
    b = Q.QuantizedB(codes=H.to_dev(w["codes"]), scales=H.to_dev(w["scales"]), params=Q.QuantParams(layout, n, k // 64),
                     mode=Q.MODE_U4 if bits == 4 else Q.MODE_U8, correction=correction, signed_codes=signed,
                     correction_data=None if w["corr"] is None else H.to_dev(w["corr"]))
    Q.MatmulKernel(w_dt, H.BF16, d_dt).encode(Q.MatmulArguments(
        a=a, b=b, d=d, m=m, n=n, k=k, d_transform=Q.MatmulDOps(ab_scale=0.5 if d_ops else 1.0, accumulate=d_ops,
                                                               bias=None if bias is None else H.to_dev(bias))))
    torch.cuda.synchronize()
    got = H.load(O, H.from_dev(d, np.float32 if d_dt == H.F32 else np.uint16), d_dt)
    vals = q.astype(np.float32)[:, [O.int8_code_index(bool(grouped), i) for i in range(k)]] * np.repeat(sc, ag, 1)
    mag = H.dequant_magnitude(O, w["codes"], w["scales"], w["corr"], n, k, bits, 64, layout, correction, w_dt,
                              vals.astype(np.float32).ravel(), H.F32, m, signed=signed, out_n=n)
    check(got, H.load(O, want, d_dt), mag=mag + (4.0 if d_ops else 0.0), label=f"m{m} n{n} k{k} b{bits}")


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("grouped", [0, 1])
@pytest.mark.parametrize("m,n,k,ag", [(1, 1, 64, 64), (3, 33, 576, 64), (16, 70, 1152, 128), (17, 40, 2112, 64),
                                      (33, 96, 1280, 128), (20, 16500, 192, 64), (70, 8300, 128, 128),
                                      (150, 5000, 320, 64)])
def test_shapes(qmm, oracle, bits, grouped, m, n, k, ag):
    _run(qmm, oracle, m, n, k, bits, ag, grouped, layout=(m + n) % 2)


# (m, n, k, activation group) and the shape (16-row blocks, waves along K): passes of 128 values a wave, at least 4 and an odd group
SHAPES = [(17, 40, 4160, 64, (1, 8)), (19, 8310, 4672, 64, (2, 8)), (17, 8310, 2112, 64, (2, 4)),
          (33, 8310, 1088, 64, (2, 2)), (50, 16510, 1088, 64, (4, 2)), (35, 33010, 576, 64, (4, 1))]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k,ag,shape", SHAPES)
def test_each_shape(qmm, oracle, bits, m, n, k, ag, shape):
    _run(qmm, oracle, m, n, k, bits, ag, grouped=bits == 8, layout=(shape[0] + shape[1]) % 2)


# one and two rows (m, n, k), and whether 4-bit and 8-bit ones take a wave a row
ROWS = [(1, 700, 2112, True, True), (1, 3200, 2112, False, False), (1, 2304, 1024, True, True), (1, 600, 576, False, True),
        (2, 500, 2112, True, False), (2, 1030, 2112, False, False), (2, 500, 832, False, True)]


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("m,n,k,wave4,wave8", ROWS)
def test_one_and_two_rows(qmm, oracle, bits, m, n, k, wave4, wave8):
    _run(qmm, oracle, m, n, k, bits, 64, grouped=n % 3 == 0, layout=(m + k // 64) % 2)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("correction,signed,w_dt", [(0, False, H.BF16), (1, True, H.F16), (0, True, H.F16)])
def test_corrections(qmm, oracle, bits, correction, signed, w_dt):
    _run(qmm, oracle, 21, 75, 704, bits, 64, 1, 0, correction, signed, w_dt)


def test_d_ops(qmm, oracle):
    _run(qmm, oracle, 5, 45, 832, 4, 64, 1, 1, d_ops=True)
    _run(qmm, oracle, 40, 300, 832, 8, 64, 0, 1, d_dt=H.BF16, d_ops=True)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("k", [1088, 4096, 12288])
def test_few_rows_round_as_one_row_a_wave(qmm, bits, k):
    """The f32 sums of up to 16 rows against the 64-bit product. Sums of t terms
    in p parallel partial sums that meet in a tree have a relative 2-norm error
    of about 0.4 * 2^-24 * sqrt(t / (2 p) + log2 p + 2) (independent roundings
    of 0.4 ulp on average; the 2 for the term's own): with t = k / 32 groups'
    pieces on the 64 lanes that one wave a row has, 8.9e-8 at 12288. Measured
    6 to 9.6e-8 for that form, and 1.2 to 1.9e-7 where eight waves add
    uncentred terms one by one: the bar is 1.05e-7."""
    g = torch.Generator(device="cuda").manual_seed(k + bits)
    n, m, top = 512, 16, 1 << bits
    codes = torch.randint(0, top, (n, k), generator=g, device="cuda", dtype=torch.uint8)
    s = (0.002 + 0.002 * torch.rand(n, k // 64, generator=g, device="cuda")).to(torch.bfloat16)
    b = (-s.float() * top / 2 * (0.95 + 0.1 * torch.rand(n, k // 64, generator=g, device="cuda"))).to(torch.bfloat16)
    q = torch.randint(-127, 128, (m, k), generator=g, device="cuda").to(torch.int8)
    sa = 0.001 + 0.01 * torch.rand(m, k // 64, generator=g, device="cuda")
    d = torch.zeros(m, n, device="cuda")
    packed = (codes[:, 0::2] | (codes[:, 1::2] << 4)).contiguous() if bits == 4 else codes
    qmm.MatmulKernel(H.BF16, H.BF16, H.F32).encode(qmm.MatmulArguments(
        a=qmm.Int8SymmetricA(values=q, scales=sa, scale_group_size=64, code_layout=qmm.SEQUENTIAL),
        b=qmm.QuantizedB(codes=packed, scales=s, correction_data=b, params=qmm.QuantParams(0, n, k // 64),
                         mode=qmm.MODE_U4 if bits == 4 else qmm.MODE_U8), d=d, m=m, n=n, k=k))
    torch.cuda.synchronize()
    w = codes.double().view(n, -1, 64) * s.double().unsqueeze(2) + b.double().unsqueeze(2)
    want = (q.double().view(m, -1, 64) * sa.double().unsqueeze(2)).view(m, k) @ w.view(n, k).t().contiguous()
    assert ((d.double() - want).norm() / want.norm()).item() < 1.05e-7


def test_rows_in_one_call_do_not_meet(qmm, oracle):
    """Few and many rows in one call: each as alone, bit for bit (the few ones
    keep their own shape, and neither holds the other on a kernel that it would
    not take)."""
    rng = np.random.default_rng(11)
    kern = qmm.MatmulKernel(H.BF16, H.BF16, H.F32)
    args, outs = [], []
    for m, n, k in ((5, 300, 1088), (300, 2200, 1088)):
        w = H.affine_weights(oracle, rng, n, k, 4, 64, 1, 1, H.BF16)
        a = qmm.Int8SymmetricA(values=H.to_dev(rng.integers(-127, 128, (m, k)).astype(np.int8)),
                               scales=H.to_dev(rng.uniform(0.01, 0.1, (m, k // 64)).astype(np.float32)),
                               scale_group_size=64, code_layout=qmm.SEQUENTIAL)
        b = qmm.QuantizedB(codes=H.to_dev(w["codes"]), scales=H.to_dev(w["scales"]), params=qmm.QuantParams(1, n, k // 64),
                           correction_data=H.to_dev(w["corr"]))
        for _ in range(2):
            outs.append(torch.zeros(m * n, dtype=torch.float32, device="cuda"))
            args.append(qmm.MatmulArguments(a=a, b=b, d=outs[-1], m=m, n=n, k=k))
    kern.encode_many(args[0::2])
    for a in args[1::2]:
        kern.encode(a)
    torch.cuda.synchronize()
    for a, b in zip(outs[0::2], outs[1::2]):
        assert torch.equal(a, b)
