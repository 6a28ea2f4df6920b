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
