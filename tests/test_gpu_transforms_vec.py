"""Activation transforms and gated activations (8 values per thread): operands
that are not 16-byte aligned, rows of no whole number of 8 values, and in-place
rows, against the oracle bit for bit (identity gate, so no device libm); biases of
every plane type after a product's output RHT."""
import numpy as np
import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu
F32, BF16 = H.F32, H.BF16


def _shifted(a, shift):
    """The array on the device, its first element `shift` elements past an aligned address."""
    t = H.to_dev(np.concatenate([np.zeros(shift, a.dtype), a]))
    return t[shift:]


def _bits(t):
    return t.cpu().numpy().view(np.uint8)


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("shift", [0, 1, 2])
@pytest.mark.parametrize("group", [32, 64, 128])
def test_quantize_alignment(qmm, oracle, dt, shift, group):
    rng = np.random.default_rng(shift + group + dt)
    batch, count = 3, 384
    x = H.store(oracle, rng.normal(0, 1, batch * count).astype(np.float32), dt)
    f = rng.choice([-1, 1], count).astype(np.int32)
    wq, ws, wsum = oracle.activation_transform(x, f, batch, count, oracle.QUANTIZE_WITH_GROUP_SUMS, t_dt=dt,
                                               scale_group=group, sum_group=32, grouped=bool(shift & 1))
    q = qmm.ActivationQuantization.new(group, 32, True, shift & 1)
    gq = torch.zeros(batch * count + shift, dtype=torch.int8, device="cuda")[shift:]
    gs = torch.zeros(batch * count // group, dtype=torch.float32, device="cuda")
    gsum = torch.zeros(batch * count // 32, dtype=torch.int32, device="cuda")
    qmm.ActivationTransform.quantize(dt, q).encode_quantize(_shifted(x, shift), gq, gs, gsum, _shifted(f, shift), batch,
                                                            count)
    torch.cuda.synchronize()
    assert np.array_equal(gq.cpu().numpy(), wq)
    assert np.array_equal(gs.cpu().numpy().view(np.uint32), ws.view(np.uint32))
    assert np.array_equal(gsum.cpu().numpy(), wsum)


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("shift", [0, 1])
def test_output_rht_alignment(qmm, oracle, dt, shift):
    rng = np.random.default_rng(shift + dt)
    batch, count = 2, 96
    x = H.store(oracle, rng.normal(0, 1, batch * count).astype(np.float32), dt)
    f = rng.choice([-1, 1], count).astype(np.int32)
    bias = H.store(oracle, rng.normal(0, 1, count).astype(np.float32), dt)
    want = oracle.activation_transform(x, f, batch, count, oracle.OUTPUT_RHT, t_dt=dt, bias=bias, bias_dt=dt)
    d = _shifted(x, shift)
    qmm.ActivationTransform.output_rht(dt, dt, in_place=True).encode_fp_in_place(d, H.to_dev(f), _shifted(bias, shift),
                                                                                batch, count)
    torch.cuda.synchronize()
    assert np.array_equal(_bits(d), np.asarray(want).view(np.uint8))


@pytest.mark.parametrize("w_dt", [F32, H.F16, BF16])
@pytest.mark.parametrize("d_dt", [F32, BF16])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("family", ["affine", "dense", "a8"])
def test_product_rht_bias_types(qmm, oracle, family, shift, d_dt, w_dt):
    """The bias after a product's output RHT has the type of the planes: the
    result is the one without a bias (as stored) plus the bias, whatever its
    type and alignment."""
    rng = np.random.default_rng(shift + d_dt + w_dt)
    m, n, k = 3, 64, 128
    f = H.to_dev(rng.choice([-1, 1], n).astype(np.int32))
    bias = H.store(oracle, rng.normal(0, 1, n).astype(np.float32), w_dt)
    x = H.to_dev(H.activations(oracle, rng, m, k, BF16))
    if family == "dense":
        b = qmm.FullPrecisionB(values=H.to_dev(H.store(oracle, rng.normal(0, 0.1, n * k).astype(np.float32), w_dt)))
    else:
        w = H.affine_weights(oracle, rng, n, k, 4, 64, 1, 1, w_dt)
        b = qmm.QuantizedB(codes=H.to_dev(w["codes"]), scales=H.to_dev(w["scales"]), params=qmm.QuantParams(1, n, k // 64),
                           correction_data=H.to_dev(w["corr"]))
    if family == "a8":
        x = qmm.Int8SymmetricA(values=H.to_dev(rng.integers(-127, 128, (m, k)).astype(np.int8)),
                               scales=H.to_dev(rng.uniform(0.01, 0.1, (m, k // 64)).astype(np.float32)),
                               scale_group_size=64, code_layout=qmm.SEQUENTIAL)
    kern = qmm.MatmulKernel(w_dt, BF16, d_dt)

    def run(bias):
        d = torch.zeros(m * n, dtype=torch.float32 if d_dt == F32 else torch.int16, device="cuda")
        kern.encode(qmm.MatmulArguments(a=x, b=b, d=d, m=m, n=n, k=k,
                                        d_transform=qmm.MatmulDOps(rht_factors=f, bias=bias)))
        torch.cuda.synchronize()
        return d

    plain = H.load(oracle, H.from_dev(run(None), np.float32 if d_dt == F32 else np.uint16), d_dt).astype(np.float32)
    want = H.store(oracle, plain + np.tile(H.load(oracle, bias, w_dt).astype(np.float32), m), d_dt)
    assert np.array_equal(_bits(run(_shifted(bias, shift))), np.asarray(want).view(np.uint8))


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("gated,offset,stride", [(40, 0, 40), (33, 5, 50), (64, 3, 80), (64, 8, 96)])
def test_gated_rows(qmm, oracle, dt, gated, offset, stride):
    """Separate operands: value rows at an offset and stride of their own (few values: one a thread)."""
    _gated(qmm, oracle, dt, 5, gated, offset, stride)


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("offset,stride", [(0, 4104), (8, 4120), (3, 4109)])
def test_gated_many_values(qmm, oracle, dt, offset, stride):
    """Past 3072 values a CU eight a thread, aligned and not."""
    batch, gated = 200, 4104
    assert batch * gated > 3072 * torch.cuda.get_device_properties(0).multi_processor_count
    _gated(qmm, oracle, dt, batch, gated, offset, stride)


def _gated(qmm, oracle, dt, batch, gated, offset, stride):
    rng = np.random.default_rng(gated + offset)
    gate = rng.normal(0, 2, batch * gated).astype(np.float32)
    value = rng.normal(0, 2, offset + batch * stride).astype(np.float32)
    g, v = H.store(oracle, gate, dt), H.store(oracle, value, dt)
    out = torch.zeros(batch * gated, dtype=torch.float32 if dt == F32 else torch.int16, device="cuda")
    qmm.GatedActMul.full_precision(dt, False, False).encode_fp(H.to_dev(g), H.to_dev(v), out, None, gated, batch, offset,
                                                              stride, qmm.ACT_IDENTITY)
    torch.cuda.synchronize()
    gf = H.load(oracle, g, dt).astype(np.float32).reshape(batch, gated)
    idx = offset + np.arange(batch)[:, None] * stride + np.arange(gated)[None, :]
    want = H.store(oracle, (H.load(oracle, v, dt).astype(np.float32)[idx] * gf).ravel(), dt)
    assert np.array_equal(_bits(out), np.asarray(want).view(np.uint8))
