"""Rows per m-tile chosen from the average rows of a routed expert: both sides of every line of
the rule (int8: 8 rows, and 24 for experts of this size; fp16 up to 128 tokens: 1 row, 2 rows
above 64 tokens or 3 with a heavy shared expert, 8 rows up to 64), on both weight layouts.  The
fp16 / int8 bar of the block's other parity tests: max abs 2e-2 against the fp32 evaluation with
the same (dequantised) weights; routing tables bit for bit."""
import numpy as np
import pytest

from _cases import spec_for
from moe_mi355x import _lib
from moe_mi355x import synthetic as syn
from moe_mi355x.device_layer import DeviceMoeLayer
from moe_mi355x.quantize import quantize_moe_tensors
from oracle import moe_oracle as orc
from test_gpu_parity import LOWP_ABS, check_routing, run_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wdt,E,k,T,m_blk,frag", [
    ("int8", 32, 4, 64, 16, True), ("int8", 32, 4, 65, 32, False), ("int8", 16, 4, 96, 32, True),
    ("int8", 16, 4, 97, 128, True), ("int8", 8, 4, 48, 32, False), ("int8", 8, 4, 49, 64, True),
    ("int8", 64, 2, 257, 32, False), ("int8", 8, 2, 33, 32, True),
    ("float16", 68, 2, 34, 16, True), ("float16", 64, 2, 33, 32, False),
    ("float16", 16, 2, 64, 32, True), ("float16", 16, 4, 34, 64, False),
    ("float16", 96, 2, 96, 32, True), ("float16", 96, 2, 97, 128, True),
    ("float16", 32, 1, 96, 32, True), ("float16", 32, 1, 97, 128, False),  # heavy shared expert
    ("float16", 200, 2, 128, 32, True), ("float16", 200, 2, 129, 128, True),
    ("float16", 200, 2, 100, 16, False)])
def test_tile_rows(mi355x, stream, wdt, E, k, T, m_blk, frag):
    print(f"[gpu] tile rows {wdt} E={E} k={k} T={T} frag={frag}", flush=True)
    shape = syn.MoeShape(syn.GLM, 128, E, k, 128, 128 if k == 1 else 64, 2.5, 1e-5)
    base = syn.make_tensors(shape, 300 + T, norm_noise=0.1)
    if wdt == "int8":
        t = quantize_moe_tensors(base)
    else:
        t = {n: (v.astype(np.float16) if n.startswith(("mlp.experts.", "mlp.shared_experts."))
                 else v) for n, v in base.items()}
    x = syn.make_inputs(301 + T, T, shape.hidden)
    spec = spec_for(shape, orc.SIGMOID_SELECT_BIAS)
    out, views = run_device(mi355x, stream, t, shape, spec, x, frag=frag)
    assert views["m_blk"] == m_blk
    ref = orc.moe_block(x, t, spec)
    check_routing(views, ref, ref["logits"], t["mlp.gate.e_score_correction_bias"], spec,
                  f"{wdt} T={T}", x, t)
    assert float(np.max(np.abs(out - ref["out"]))) <= LOWP_ABS


def test_reserved_once_serves_shorter_batches(mi355x, stream):
    """513 tokens take one router slice less than 512: buffers reserved for 513 run 512."""
    print("[gpu] reserve 513 tokens, run 512", flush=True)
    shape = syn.MoeShape(syn.QWEN, 2048, 512, 2, 32, 32, 1.0, 1e-6, has_bias=False,
                         has_shared_gate=True)
    layer = DeviceMoeLayer.synthetic(mi355x, shape, 77, stream, weight_dtype="float16",
                                     param_dtype="float32")
    cfg = layer.config(top_k=2, router_mode=_lib.MX_ROUTER_SOFTMAX, routed_scaling=1.0, eps=1e-6)
    x = syn.make_inputs(78, 513, shape.hidden)
    try:
        layer.prepare(cfg, 513)
        got = layer.forward_numpy(cfg, x[:512])
        fresh = DeviceMoeLayer.synthetic(mi355x, shape, 77, stream, weight_dtype="float16",
                                         param_dtype="float32")
        try:
            want = fresh.forward_numpy(cfg, x[:512])
        finally:
            fresh.close()
    finally:
        layer.close()
    assert np.array_equal(got, want)
