"""Projections of short inputs (``mx_proj.hip``) inside the attention blocks, against float64
products of the device's own fp16 activations.

Sizes where the kernel can go wrong: token counts at the edges of its 16-row tiles, row
counts that are no multiple of its 16- and 32-column tiles (one of them leading to rows that
are not 16-byte aligned), reduction lengths with a partial last chunk, and a reduction long
enough to be split over grid slices.  Bound: the products of fp16 (int8) pairs are exact in
fp32, so only the fp32 sums round: at most (K + 16) 2^-24 of the sum of magnitudes, plus the
row scale's multiplication for int8."""
import numpy as np
import pytest

from moe_mi355x import synthetic as syn
from moe_mi355x.full_attn import DeviceFullAttnLayer
from moe_mi355x.linear_attn import DeviceLinearAttnLayer
from moe_mi355x.moe import read_device
from moe_mi355x.quantize import quantize_rows_int8
from oracle import full_attn_oracle as fa
from oracle import linear_attn_oracle as la

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mi355x():
    from moe_mi355x.backends import MI355XBackend

    return MI355XBackend(0)


@pytest.fixture(scope="module")
def stream(mi355x):
    s = mi355x.create_stream("test-proj")
    yield s
    mi355x.destroy_stream(s)


def _weights(t, names, wdt):
    """Quantises ``names`` in place for int8; returns name -> (values, row scale), float64."""
    out = {}
    for n in names:
        if wdt == "int8":
            t[n], t[n + "_scale"] = quantize_rows_int8(t[n].astype(np.float32))
            out[n] = (t[n].astype(np.float64), t[n + "_scale"].astype(np.float64)[:, None])
        else:
            out[n] = (t[n].astype(np.float64), 1.0)
    return out


def _check(name, got, a, weight):
    w, scale = weight
    k = a.shape[1]
    want = a @ (w * scale).T
    bound = ((k + 16) * 2.0 ** -24 + 2.0 ** -23) * (np.abs(a) @ (np.abs(w) * scale).T) + 1e-30
    worst = float(np.max(np.abs(got - want) / bound))
    print(f"    {name} K={k}: worst error {worst:.3f} of the bound", flush=True)
    assert worst <= 1.0, name


@pytest.mark.parametrize("wdt", ["float16", "int8"])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 32, 33, 64])
def test_linear_attention_projections(mi355x, stream, wdt, T):
    # qkvz 3 * 2 * (32 + 512) = 3264 rows of 208, ba 99 rows, out 208 rows of 1536 (sliced)
    shape = syn.LinearAttnShape(208, 3, 32, 512, 4, 1e-6)
    print(f"[gpu] linear attention projections {wdt} T={T}", flush=True)
    t = syn.make_linear_attn_tensors(shape, 90 + T, weight_dtype=np.float16, norm_noise=0.1)
    w = _weights(t, (la.QKVZ, la.BA, la.OUT), wdt)
    x = syn.make_inputs(91 + T, T, shape.hidden)
    layer = DeviceLinearAttnLayer.from_host(mi355x, t, stream)
    try:
        out = layer.forward_numpy(x, shape.eps)
        v = layer.runner.views(layer.desc(shape.eps), T)

        def read(p, dt, n):
            return read_device(mi355x, p, dt, T * n, stream).reshape(T, n).astype(np.float64)

        vd = shape.n_heads * shape.head_dim_v
        h, act = read(v.h16, np.float16, shape.hidden), read(v.act, np.float16, vd)
        qkvz, ba = read(v.qkvz, np.float32, shape.qkvz_rows), read(v.ba, np.float32, shape.ba_rows)
        y = read(v.y, np.float32, shape.hidden)
    finally:
        layer.close()
    _check("qkvz", qkvz, h, w[la.QKVZ])
    _check("ba", ba, h, w[la.BA])
    _check("out", y, act, w[la.OUT])
    assert np.array_equal(out, x + y.astype(np.float32))


@pytest.mark.parametrize("wdt", ["float16", "int8"])
@pytest.mark.parametrize("T", [1, 16, 31, 48, 64])
def test_full_attention_projections(mi355x, stream, wdt, T):
    # q 2 * 6 * 20 = 240 rows of 272, k and v 40 rows, o 272 rows of 120 / int8 6 * 24 = 144
    hd = 20 if wdt == "float16" else 24
    s = syn.FullAttnShape(272, 6, 2, hd, 0.5, 10000.0, 1e-6)
    print(f"[gpu] full attention projections {wdt} T={T}", flush=True)
    t = syn.make_full_attn_tensors(s, 70 + T, weight_dtype=np.float16, norm_noise=0.1)
    w = _weights(t, (fa.Q, fa.K, fa.V, fa.O), wdt)
    x = syn.make_inputs(71 + T, T, s.hidden)
    layer = DeviceFullAttnLayer.from_host(mi355x, t, s.n_heads, s.n_kv_heads, s.head_dim,
                                          s.rotary_dim, s.rope_theta, stream)
    try:
        out = layer.forward_numpy(x, s.eps)
        v = layer.runner.views(layer.desc(s.eps), T)

        def read(p, dt, n):
            return read_device(mi355x, p, dt, T * n, stream).reshape(T, n).astype(np.float64)

        od, kw = s.n_heads * s.head_dim, s.n_kv_heads * s.head_dim
        h, act = read(v.h16, np.float16, s.hidden), read(v.act, np.float16, od)
        gate = read(v.qg, np.float32, 2 * od)[:, od:]
        vv, y = read(v.v, np.float32, kw), read(v.y, np.float32, s.hidden)
    finally:
        layer.close()
    # q and k are normalised and rotated in place after the projection; the gate half of the
    # q projection and v are left as they were
    wq, sq = w[fa.Q]
    _check("gate", gate, h, (wq[od:], sq[od:] if wdt == "int8" else sq))
    _check("v", vv, h, w[fa.V])
    _check("o", y, act, w[fa.O])
    assert np.array_equal(out, x + y.astype(np.float32))


@pytest.mark.parametrize("wdt,hidden,heads,dk,dv,T", [
    ("float16", 192, 9, 32, 256, 65),    # out: 36 stages in 4 slices, one row past 64
    ("float16", 192, 9, 32, 256, 129),   # two row tiles
    ("float16", 2048, 9, 32, 64, 300),   # out: 9 stages, one slice; two blocks per CU
    ("float16", 128, 8, 32, 264, 128),   # out: 33 stages in 4 slices, the last one shorter
    ("int8", 384, 9, 32, 256, 65),       # out: 18 stages in 4 slices, the last one shorter
    ("int8", 128, 4, 32, 1056, 129),     # out: 33 stages in 7 slices (8 would leave one empty)
    ("int8", 128, 32, 128, 128, 1100),   # qkvz on 128 x 256 tiles, the rest on 128 x 128
    ("int8", 256, 4, 32, 24, 70),        # out: reduction 96, on the grouped kernels
])
def test_linear_attention_gemm(mi355x, stream, wdt, hidden, heads, dk, dv, T):
    shape = syn.LinearAttnShape(hidden, heads, dk, dv, 4, 1e-6)
    print(f"[gpu] dense GEMM {wdt} hidden {hidden} vd {heads * dv} T={T}", flush=True)
    t = syn.make_linear_attn_tensors(shape, 50 + T, weight_dtype=np.float16, norm_noise=0.1)
    w = _weights(t, (la.QKVZ, la.BA, la.OUT), wdt)
    x = syn.make_inputs(51 + T, T, hidden)
    layer = DeviceLinearAttnLayer.from_host(mi355x, t, stream)
    try:
        out = layer.forward_numpy(x, shape.eps)
        v = layer.runner.views(layer.desc(shape.eps), T)

        def read(p, dt, n):
            return read_device(mi355x, p, dt, T * n, stream).reshape(T, n).astype(np.float64)

        h, act = read(v.h16, np.float16, hidden), read(v.act, np.float16, heads * dv)
        qkvz, ba = read(v.qkvz, np.float32, shape.qkvz_rows), read(v.ba, np.float32, shape.ba_rows)
    finally:
        layer.close()
    _check("qkvz", qkvz, h, w[la.QKVZ])
    _check("ba", ba, h, w[la.BA])
    # out = x + act W^T: one more rounding, of a sum no larger than |x| + the magnitudes
    wo = w[la.OUT][0] * w[la.OUT][1]
    k = act.shape[1]
    bound = ((k + 16) * 2.0 ** -24 + 2.0 ** -23) * (np.abs(act) @ np.abs(wo).T + np.abs(x)) + 1e-30
    worst = float(np.max(np.abs(out - (x + act @ wo.T)) / bound))
    print(f"    out K={k}: worst error {worst:.3f} of the bound", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("T", [16, 17, 24, 32])
def test_wide_fp16_products(mi355x, stream, T):
    """qkvz and ba of 20,512 columns in all: on k_proj up to 16 tokens, on the GEMM from 17 (its
    128-row tiles mostly padding), while the narrow out projection stays on k_proj."""
    shape = syn.LinearAttnShape(128, 32, 128, 128, 4, 1e-6)
    print(f"[gpu] wide fp16 projections T={T}", flush=True)
    t = syn.make_linear_attn_tensors(shape, 60 + T, weight_dtype=np.float16, norm_noise=0.1)
    w = _weights(t, (la.QKVZ, la.BA, la.OUT), "float16")
    x = syn.make_inputs(61 + T, T, shape.hidden)
    layer = DeviceLinearAttnLayer.from_host(mi355x, t, stream)
    try:
        out = layer.forward_numpy(x, shape.eps)
        v = layer.runner.views(layer.desc(shape.eps), T)

        def read(p, dt, n):
            return read_device(mi355x, p, dt, T * n, stream).reshape(T, n).astype(np.float64)

        h, act = read(v.h16, np.float16, 128), read(v.act, np.float16, 4096)
        qkvz, ba = read(v.qkvz, np.float32, shape.qkvz_rows), read(v.ba, np.float32, shape.ba_rows)
        y = read(v.y, np.float32, 128)
    finally:
        layer.close()
    _check("qkvz", qkvz, h, w[la.QKVZ])
    _check("ba", ba, h, w[la.BA])
    _check("out", y, act, w[la.OUT])
    assert np.array_equal(out, x + y.astype(np.float32))


@pytest.mark.parametrize("kind,hidden,heads,dk,dv,T", [
    ("linear", 384, 9, 32, 256, 65),    # 4 reduction slices
    ("linear", 128, 4, 32, 1056, 129),  # 7 slices
    ("linear", 256, 4, 32, 32, 130),    # one slice, 128 x 128 tiles
    ("linear", 2048, 4, 32, 32, 2200),  # 128 x 256 tiles
    ("linear", 2048, 4, 32, 32, 4500),  # whole rounds of 128 x 256 tiles, the rest on 128 x 128
    ("full", 384, 4, 128, 128, 66),     # slices
    ("full", 256, 4, 32, 32, 200),      # one slice
])
def test_int8_product_view_of_long_inputs(mi355x, stream, kind, hidden, heads, dk, dv, T):
    """The view y holds the whole product act W^T for int8 weights at every length, however the
    GEMM forms out = x + y."""
    print(f"[gpu] int8 y view, {kind} hidden {hidden} K {heads * dv} T={T}", flush=True)
    x = syn.make_inputs(31 + T, T, hidden)
    if kind == "linear":
        shape = syn.LinearAttnShape(hidden, heads, dk, dv, 4, 1e-6)
        t = syn.make_linear_attn_tensors(shape, 30 + T, weight_dtype=np.float16, norm_noise=0.1)
        w = _weights(t, (la.QKVZ, la.BA, la.OUT), "int8")[la.OUT]
        layer = DeviceLinearAttnLayer.from_host(mi355x, t, stream)
    else:
        s = syn.FullAttnShape(hidden, heads, 2, dk, 0.25, 10000.0, 1e-6)
        t = syn.make_full_attn_tensors(s, 30 + T, weight_dtype=np.float16, norm_noise=0.1)
        w = _weights(t, (fa.Q, fa.K, fa.V, fa.O), "int8")[fa.O]
        layer = DeviceFullAttnLayer.from_host(mi355x, t, heads, 2, dk, s.rotary_dim, s.rope_theta,
                                              stream)
    try:
        out = layer.forward_numpy(x, 1e-6)
        v = layer.runner.views(layer.desc(1e-6), T)
        act = read_device(mi355x, v.act, np.float16, T * heads * dv, stream).reshape(T, -1)
        y = read_device(mi355x, v.y, np.float32, T * hidden, stream).reshape(T, hidden)
    finally:
        layer.close()
    _check("out", y.astype(np.float64), act.astype(np.float64), w)
    # the sum with x, rounded once
    assert np.all(np.abs(out - (x.astype(np.float64) + y)) <= 2.0 ** -23 * (np.abs(x) + np.abs(y)))


def test_workspace_never_shrinks_with_tokens(mi355x):
    """A workspace sized for a batch serves every shorter one (the executors size it once)."""
    from moe_mi355x import _lib
    from moe_mi355x.full_attn import workspace_bytes as fa_bytes
    from moe_mi355x.linear_attn import workspace_bytes as la_bytes

    for wdt in (_lib.MX_DT_F32, _lib.MX_DT_F16, _lib.MX_DT_I8):
        for hidden, n, dk, dv in ((2048, 32, 128, 128), (192, 9, 32, 256), (8192, 4, 64, 64)):
            d = _lib.MxLinearAttnDesc(hidden, n, dk, dv, 4, wdt, _lib.MX_DT_F32, 1e-6)
            sizes = [la_bytes(d, T) for T in range(1, 700)]
            assert sizes == sorted(sizes)
            f = _lib.MxFullAttnDesc(hidden, n, 1, dk, dk // 2, wdt, _lib.MX_DT_F32, 1e4, 1e-6)
            sizes = [fa_bytes(f, T) for T in range(1, 700)]
            assert sizes == sorted(sizes)
