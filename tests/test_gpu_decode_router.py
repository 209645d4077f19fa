"""Router and dispatch of 5 to 64 tokens: token counts on both sides of one token per wave of the
one-workgroup form (16, 8 above 512 experts) and of two with at most 64 experts, expert counts on
both sides of the lines for 1, 2 and 4 expert rows per block (512 and 1024 blocks of one row), with
rows left over (513 rows), and around whole waves of the dispatch scan.  Selections by the routing rules of the other parity
tests, integer tables bit for bit, outputs to the block's fp32 bar (1e-4 normwise).  k stays small
beside E: the selection gaps of many experts shrink below the tie rule's 1e-5 otherwise."""
import numpy as np
import pytest

from _cases import normwise_err, spec_for
from moe_mi355x import synthetic as syn
from oracle import moe_oracle as orc
from test_gpu_parity import FP32_REL, check_routing, run_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,k,T,gate", [
    (512, 10, 5, True), (512, 10, 8, True), (512, 4, 16, True), (512, 10, 17, True),
    (512, 10, 64, True), (160, 8, 16, False), (160, 8, 17, False), (160, 8, 25, False),
    (160, 8, 64, False), (64, 3, 33, False), (64, 3, 32, True), (64, 4, 17, False), (32, 2, 24, True),
    (65, 4, 16, True), (96, 4, 17, False), (63, 5, 64, True), (65, 4, 18, False),
    (520, 6, 8, False), (520, 6, 9, True), (1024, 6, 33, False), (130, 12, 64, True),
    (5, 5, 40, True), (1, 1, 20, False)])
def test_decode_router(mi355x, stream, E, k, T, gate):
    print(f"[gpu] decode router E={E} k={k} T={T} gate={gate}", flush=True)
    shape = syn.MoeShape(syn.QWEN if gate else syn.GLM, 264, E, k, 32, 32, 1.0 if gate else 2.5,
                         1e-5, has_bias=not gate, has_shared_gate=gate)
    t = syn.make_tensors(shape, 500 + T, norm_noise=0.1)
    x = syn.make_inputs(501 + T, T, shape.hidden)
    spec = spec_for(shape, orc.SOFTMAX if gate else orc.SIGMOID_SELECT_BIAS)
    out, views = run_device(mi355x, stream, t, shape, spec, x)
    ref = orc.moe_block(x, t, spec)
    check_routing(views, ref, ref["logits"], None if gate else
                  t["mlp.gate.e_score_correction_bias"], spec, f"E={E} T={T}", x, t)
    assert normwise_err(out, ref["out"]) <= FP32_REL
