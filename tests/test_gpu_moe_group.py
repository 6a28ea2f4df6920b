"""Routed experts of prompts (more than 16 tokens, group-64 banks): slots of up
to 64 routes. Edges of the slots (17, 33 and 49 routes of an expert, more than
64), of the column tiles (rows that fill no whole workgroup or wave) and of K
(one chunk, odd group counts), against the oracle; bit-exact weights through
one-hot rows; signed codes against the same unsigned ones."""
import numpy as np
import pytest
import torch

from tests import helpers as H
from tests import test_gpu_moe as G
from tests import test_gpu_moe_exact as X
from tests.moe_cases import case

pytestmark = pytest.mark.gpu


SLOTS = [(17, 256, 192, 8, 2, True), (40, 64, 64, 2, 2, True), (70, 320, 64, 2, 1, False),
         (150, 192, 320, 3, 2, True), (49, 512, 576, 1, 1, True)]
EXACT = [(20, 320, 192, 4), (130, 256, 128, 2), (48, 640, 448, 1)]


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("rows,model,hidden,experts,active,biased", SLOTS)
def test_prompt_slots(qmm, oracle, rows, model, hidden, experts, active, biased, layout):
    c = case(oracle, 31 * rows + model + layout, rows, model, hidden, experts, active, layout=layout, biased=biased)
    G.routed_check(qmm, oracle, c)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("rows,model,hidden,experts", EXACT)
def test_prompt_products_exact(qmm, oracle, rows, model, hidden, experts, layout):
    X.test_routed_up_product_exact(qmm, oracle, rows, model, hidden, experts, layout)
    X.test_routed_down_product_exact(qmm, oracle, rows, model, hidden, experts, layout)


@pytest.mark.parametrize("rows", [33, 64])
def test_one_expert_of_few_tokens(qmm, oracle, rows):
    """Left to the slot form by the rule."""
    G.routed_check(qmm, oracle, case(oracle, rows, rows, 1024, 512, 1, 1, layout=1, biased=True))


def test_prompt_signed_codes(qmm, oracle):
    c = case(oracle, 5, 60, 256, 192, 3, 2)
    want = G.routed_run(qmm, c)
    args = [H.to_dev(c["x"]), H.to_dev(c["logits"])]
    for name, rows, cols in (("up", 3 * 2 * 192, 256), ("down", 3 * 256, 192)):
        b = c[name]
        args.append(qmm.QuantizedB(codes=H.to_dev(np.asarray(b["codes"], np.uint8) ^ 0x88), scales=H.to_dev(b["scales"]),
                                   correction_data=H.to_dev(b["biases"]), params=qmm.QuantParams(1, rows, cols // 64),
                                   group_size=64, signed_codes=True))
    out = qmm.routed_experts(*args, 60, 256, 192, 3, 2)
    torch.cuda.synchronize()
    got = (H.from_dev(out.view(torch.int16), np.uint16).astype(np.uint32) << 16).view(np.float32)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def _by_slots(qmm, c, step=8):
    """The same tokens, `step` a call: the slot form of few tokens."""
    rows = []
    for r in range(0, c["rows"], step):
        n = min(step, c["rows"] - r)
        part = dict(c, rows=n, x=c["x"].reshape(c["rows"], -1)[r:r + n].ravel(),
                    logits=c["logits"].reshape(c["rows"], -1)[r:r + n].ravel())
        rows.append(G.routed_run(qmm, part).reshape(n, -1))
    return np.concatenate(rows)


def test_prompt_activation_range(qmm, oracle):
    """Tokens of 2^-100 to 2^50, of mixed magnitudes and of bf16 subnormals: as
    in the slot form, whose products are the same up to the order of the f32 sums
    (a bf16 ulp in each of the three stages, of the row's largest value)."""
    c = case(oracle, 41, 60, 256, 192, 3, 2)
    rng = np.random.default_rng(41)
    x = oracle.bf16_to_f32(c["x"]).reshape(60, 256) * np.exp2(rng.integers(-100, 51, (60, 1))).astype(np.float32)
    x[1::7, :64] *= np.float32(2.0 ** -60)
    x[5] = rng.integers(1, 127, 256) * 2.0 ** -133
    c["x"] = oracle.f32_to_bf16(np.ascontiguousarray(x.astype(np.float32).ravel()))
    got, want = G.routed_run(qmm, c).reshape(60, -1).astype(np.float64), _by_slots(qmm, c).astype(np.float64)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    assert np.all(np.abs(got - want) <= 3 * 2.0 ** -8 * np.abs(want).max(axis=1, keepdims=True))
    assert (np.abs(want).max(axis=1) > 0).sum() > 40


def test_prompt_non_finite_activations(qmm, oracle):
    """Infinities and NaN stay in their token, and there as in the slot form: not finite in the same places."""
    c = case(oracle, 43, 40, 256, 192, 3, 2)
    x = oracle.bf16_to_f32(c["x"]).reshape(40, 256).copy()
    plain = G.routed_run(qmm, c).reshape(40, -1)
    x[3, 70], x[17, 5], x[30, 255], x[38, 0] = np.inf, -np.inf, np.nan, 3.3e38
    c["x"] = oracle.f32_to_bf16(np.ascontiguousarray(x.ravel()))
    got, want = G.routed_run(qmm, c).reshape(40, -1), _by_slots(qmm, c)
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    touched = [3, 17, 30, 38]
    assert not np.isfinite(got[[3, 17, 30]]).all()
    others = np.setdiff1d(np.arange(40), touched)
    assert np.array_equal(got[others].view(np.uint32), plain[others].view(np.uint32))
