"""fp16 attention of the full-attention block at the sizes where its packed operands and query
blocks can go wrong: head dims that are no power of two (padded to 32, 64, 128 or 256), token
counts at the edges of the 32-key tiles and of the query blocks, several query heads per
key/value head.  Compared with the oracle's attention in float64 over the block's own q, k, v and
gate rows.  Tolerance: q, k, v and the probabilities are rounded to fp16 (2^-11 each) before
products that are summed in fp32, and the gated output once more, five roundings in all;
normwise 4 x 2^-11 covers them."""
import numpy as np
import pytest

from moe_mi355x import synthetic as syn
from moe_mi355x.full_attn import DeviceFullAttnLayer
from moe_mi355x.moe import read_device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mi355x():
    from moe_mi355x.backends import MI355XBackend

    return MI355XBackend(0)


@pytest.fixture(scope="module")
def stream(mi355x):
    s = mi355x.create_stream("test-fa16")
    yield s
    mi355x.destroy_stream(s)


@pytest.mark.parametrize("hd,nh,nkv,T", [
    (72, 4, 2, 33), (96, 4, 1, 70), (160, 4, 2, 40), (252, 2, 1, 129), (20, 4, 2, 65),
    (256, 8, 1, 1), (256, 8, 1, 16), (256, 8, 2, 17), (256, 8, 1, 32), (256, 8, 2, 64),
    (256, 8, 2, 65), (256, 16, 2, 400), (128, 8, 2, 63), (128, 8, 1, 513), (256, 2, 2, 1030),
    # an even number of query blocks: all resident (512 blocks), and more than that with one and
    # with two query sets per wave
    (128, 16, 2, 2040), (128, 16, 2, 2170), (128, 32, 4, 2200)])
def test_attention_matches_oracle(mi355x, stream, hd, nh, nkv, T):
    s = syn.FullAttnShape(128, nh, nkv, hd, 0.25 if hd % 8 == 0 else 0.5, 10000.0, 1e-6)
    if s.rotary_dim % 2:
        s = syn.FullAttnShape(128, nh, nkv, hd, 0.0, 10000.0, 1e-6)
    print(f"[gpu] fp16 attention hd={hd} heads={nh}/{nkv} T={T}", flush=True)
    t = syn.make_full_attn_tensors(s, 20 + T, weight_dtype=np.float16, norm_noise=0.1)
    x = syn.make_inputs(21 + T, T, s.hidden)
    layer = DeviceFullAttnLayer.from_host(mi355x, t, nh, nkv, hd, s.rotary_dim, s.rope_theta,
                                          stream)
    try:
        layer.forward_numpy(x, s.eps)
        v = layer.runner.views(layer.desc(s.eps), T)
        od, kw = nh * hd, nkv * hd

        def read(p, dt, n):
            return read_device(mi355x, p, dt, T * n, stream).reshape(T, n).astype(np.float64)

        qg, act = read(v.qg, np.float32, 2 * od), read(v.act, np.float16, od)
        k, vv = read(v.k, np.float32, kw), read(v.v, np.float32, kw)
    finally:
        layer.close()
    want = np.empty((T, nh, hd))
    mask = np.triu(np.ones((T, T), bool), 1)
    for h in range(nh):
        c = slice(h * hd, (h + 1) * hd)
        kc = slice(h // (nh // nkv) * hd, (h // (nh // nkv) + 1) * hd)
        sc = np.where(mask, -np.inf, qg[:, c] @ k[:, kc].T / np.sqrt(hd))
        p = np.exp(sc - sc.max(axis=1, keepdims=True))
        want[:, h] = (p / p.sum(axis=1, keepdims=True)) @ vv[:, kc]
    want = want.reshape(T, od) / (1 + np.exp(-qg[:, od:]))
    err = np.linalg.norm(act - want) / np.linalg.norm(want)
    print(f"    normwise err {err:.2e}", flush=True)
    assert np.all(np.isfinite(act)) and err <= 4 * 2.0 ** -11


def test_norm_weights_at_any_address(mi355x, stream):
    """q / k norm weights off the 16-byte boundary take the scalar RoPE form: same block output
    up to the order of the row sums (fp32) and the fp16 roundings after them."""
    hd, nh, nkv, T = 64, 4, 2, 37
    print(f"[gpu] norm weights 4 bytes off, hd={hd} T={T}", flush=True)
    s = syn.FullAttnShape(128, nh, nkv, hd, 0.25, 10000.0, 1e-6)
    t = syn.make_full_attn_tensors(s, 7, weight_dtype=np.float16, norm_noise=0.1)
    x = syn.make_inputs(8, T, s.hidden)
    layer = DeviceFullAttnLayer.from_host(mi355x, t, nh, nkv, hd, s.rotary_dim, s.rope_theta,
                                          stream)
    raw = np.concatenate([np.zeros(1), t["self_attn.q_norm.weight"].ravel(),
                          t["self_attn.k_norm.weight"].ravel()]).astype(np.float32)
    buf = mi355x.alloc_device(raw.nbytes)
    try:
        want = layer.forward_numpy(x, s.eps)
        mi355x.copy_h2d_ptr_async(buf.handle, raw.ctypes.data, raw.nbytes, stream)
        mi355x.synchronize_stream(stream)
        w = layer.weights()
        w.q_norm_w = int(buf.handle) + 4
        w.k_norm_w = int(buf.handle) + 4 + 4 * hd
        got = layer.runner.forward_numpy(layer.desc(s.eps), w, x, stream)
    finally:
        mi355x.free_device(buf)
        layer.close()
    assert np.linalg.norm(got - want) <= 4 * 2.0 ** -11 * np.linalg.norm(want - x)
