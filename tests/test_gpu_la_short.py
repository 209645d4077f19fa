"""Conv, gates and recurrence of short inputs in one launch, against the oracle run on the
device's own projections: token counts at the edges of the 1-, 4- and 16-token forms and past
them (separate launches), key heads of 64, 128 and 256, value heads that are no multiple of a
block's 16 rows; the conv and gates of longer inputs at the edges of 4, 8 and 16 tokens per
thread.  Bounds: the fp32 conv and gates to 2e-6 normwise, the recurrence to 1e-5."""
import numpy as np
import pytest

from moe_mi355x import synthetic as syn
from moe_mi355x.linear_attn import DeviceLinearAttnLayer
from moe_mi355x.moe import read_device
from oracle import linear_attn_oracle as la

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mi355x():
    from moe_mi355x.backends import MI355XBackend

    return MI355XBackend(0)


@pytest.fixture(scope="module")
def stream(mi355x):
    s = mi355x.create_stream("test-la-short")
    yield s
    mi355x.destroy_stream(s)


def _err(got, want):
    return np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30)


def _stages(mi355x, stream, dk, dv, n, T, pdt, taps):
    """Run a layer of small hidden size; conv and gates checked, its stage buffers returned."""
    shape = syn.LinearAttnShape(64, n, dk, dv, taps, 1e-6)
    t = syn.make_linear_attn_tensors(shape, 40 + T, weight_dtype=np.float32, param_dtype=pdt,
                                     norm_noise=0.1)
    x = syn.make_inputs(41 + T, T, shape.hidden)
    layer = DeviceLinearAttnLayer.from_host(mi355x, t, stream)
    try:
        layer.forward_numpy(x, shape.eps)
        w = layer.runner.views(layer.desc(shape.eps), T)

        def read(p, cols):
            return read_device(mi355x, p, np.float32, T * cols, stream).reshape(T, cols)

        qd, vd = n * dk, n * dv
        qkvz, ba = read(w.qkvz, 2 * qd + 2 * vd), read(w.ba, qd + n)
        q, kb, v = read(w.q, qd), read(w.kb, qd), read(w.v, vd)
        decay, o = read(w.decay, n), read(w.o, vd)
    finally:
        layer.close()
    conv = la.silu(la.causal_conv1d(qkvz[:, :2 * qd + vd], t[la.CONV].squeeze(1)))
    g = -np.exp(t[la.A_LOG]) * la.softplus(ba[:, qd:] + t[la.DT_BIAS])
    for name, got, want in (("q", q, conv[:, :qd]), ("v", v, conv[:, 2 * qd:]),
                            ("kb", kb, la.sigmoid(ba[:, :qd]) * conv[:, qd:2 * qd]),
                            ("decay", decay, np.exp(g))):
        assert _err(got, want) <= 2e-6, name
    return q, kb, v, decay, o


@pytest.mark.parametrize("dk,dv,n,T,pdt", [
    (128, 128, 2, 1, np.float32), (64, 40, 3, 1, np.float16), (256, 16, 1, 1, np.float32),
    (128, 128, 2, 2, np.float16), (64, 64, 2, 4, np.float32), (256, 24, 2, 3, np.float32),
    (128, 8, 3, 5, np.float32), (64, 128, 2, 16, np.float32), (128, 128, 2, 17, np.float16),
    (256, 40, 2, 31, np.float32), (64, 20, 3, 63, np.float32), (128, 128, 1, 63, np.float32),
    (256, 64, 1, 48, np.float16)])
def test_short_inputs_match_oracle(mi355x, stream, dk, dv, n, T, pdt):
    print(f"[gpu] short linear attention dk={dk} dv={dv} heads={n} T={T}", flush=True)
    q, kb, v, decay, o = _stages(mi355x, stream, dk, dv, n, T, pdt, 4)
    want = la.gated_recurrence(q, kb, v, np.log(decay), n, dk, dv)
    err = _err(o, want)
    print(f"    recurrence normwise err {err:.2e}", flush=True)
    assert err <= 1e-5


@pytest.mark.parametrize("T", [160, 161, 1535, 1537])
@pytest.mark.parametrize("taps,pdt", [(4, np.float32), (4, np.float16), (3, np.float32)])
def test_conv_of_long_inputs(mi355x, stream, T, taps, pdt):
    print(f"[gpu] linear attention conv taps={taps} T={T}", flush=True)
    _stages(mi355x, stream, 32, 24, 2, T, pdt, taps)
