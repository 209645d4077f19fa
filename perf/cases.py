"""The calls that perf measurements of this package make.

Four kinds of call, each through the package's public entry points on torch-owned device
memory and the current stream, the way a program that keeps its layers in HBM uses it:

  "moe"     one MoE block (RMSNorm, router, top-k, experts, combine): MoeRunner.forward_device
  "linear"  one Qwen3-Next linear-attention block: LinearAttnRunner.forward_device
  "full"    one Qwen3-Next gated full-attention block: FullAttnRunner.forward_device
  "stack"   four resident Qwen3-Next layers (three linear-attention, one full-attention, each
            with its MoE block) through OffloadRuntime and Qwen3NextExecutor, NumPy in and out

Shapes are the package's own workload shapes (moe_mi355x.synthetic): GLM-4.7-sized and
Qwen3-Next-sized layers.  ``tokens`` runs from one token (a decode step) over small decode
batches and short prompts to the longest prefill of the benchmark.  Expert and projection
weights are fp16 or per-row int8; parameters (norms, router, conv taps) are fp32.
"""
from __future__ import annotations

import math
import os
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("disk-mem-off_amd"))

from moe_mi355x import _lib, synthetic as syn  # noqa: E402
from moe_mi355x.backends import MI355XBackend  # noqa: E402
from moe_mi355x.device_layer import DeviceMoeLayer  # noqa: E402
from moe_mi355x.executors import Qwen3NextExecutor  # noqa: E402
from moe_mi355x.full_attn import FullAttnLayout, FullAttnRunner  # noqa: E402
from moe_mi355x.layout import MoeLayerLayout, make_layer_spec  # noqa: E402
from moe_mi355x.linear_attn import LinearAttnLayout, LinearAttnRunner  # noqa: E402
from moe_mi355x.moe import MoeConfig, MoeRunner, tile_experts  # noqa: E402
from moe_mi355x.runtime import OffloadRuntime  # noqa: E402
from moe_mi355x.scheduler import LookaheadScheduler  # noqa: E402
from moe_mi355x.storage import DeviceResidentStorage  # noqa: E402
from moe_mi355x.types import DeviceBuffer  # noqa: E402

SHAPES = {"glm": syn.GLM47, "qwen": syn.QWEN3_NEXT}
LA = syn.QWEN3_NEXT_LINEAR
FA = syn.QWEN3_NEXT_FULL
STACK_KINDS = ("linear", "linear", "linear", "full")  # Qwen3-Next: every fourth layer is full
TORCH = {"float32": torch.float32, "float16": torch.float16, "int8": torch.int8}
ESZ = {"float32": 4, "float16": 2, "int8": 1}
ALIGN = 256


def _moe(name, shape, tokens, dtype="float16", layout="frag16", skew=0.0):
    return {"name": name, "kind": "moe", "shape": shape, "tokens": tokens, "dtype": dtype,
            "layout": layout, "skew": skew}


def listed():
    return [
        # One token through a small-expert MoE block: the latency of a single user's decode.
        _moe("moe_qwen_1", "qwen", 1),
        # A decode batch on large experts (the benchmark's headline).
        _moe("moe_glm_32", "glm", 32),
        # A decode batch on per-row int8 experts, the format that halves the weight bytes.
        _moe("moe_glm_int8_16", "glm", 16, dtype="int8"),
        # A short prompt, of no round length: between the decode batches and the long prefills.
        _moe("moe_qwen_200", "qwen", 200),
        # The benchmark's long Qwen3-Next prefill.
        _moe("moe_qwen_4096", "qwen", 4096),
        # A long prefill with uneven expert loads (from about 0 to 300 rows each).
        _moe("moe_glm_2048", "glm", 2048, skew=0.04),
        # One decode token through a linear-attention block: launches and weight streaming.
        {"name": "linear_1", "kind": "linear", "tokens": 1, "dtype": "float16"},
        # A prompt of ordinary length on int8 projections.
        {"name": "linear_int8_300", "kind": "linear", "tokens": 300, "dtype": "int8"},
        # A long prefill through the linear-attention block.
        {"name": "linear_4096", "kind": "linear", "tokens": 4096, "dtype": "float16"},
        # An ordinary prompt of odd length through the full-attention block.
        {"name": "full_777", "kind": "full", "tokens": 777, "dtype": "float16"},
        # A long prefill, where attention itself is a third of the block.
        {"name": "full_4096", "kind": "full", "tokens": 4096, "dtype": "float16"},
        # A small batch through four whole layers, as the offload runtime drives them.
        {"name": "stack_24", "kind": "stack", "tokens": 24, "dtype": "float16"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "linear", "full"])
    dtype = rng.choice(["float16", "float16", "int8"])
    if kind == "moe":
        shape = rng.choice(["glm", "qwen"])
        return {"kind": kind, "shape": shape,
                "tokens": _log_int(rng, 1, 2048 if shape == "glm" else 4096), "dtype": dtype,
                "layout": rng.choice(["frag16", "frag16", "rows"]),
                "skew": rng.choice([0.0, 0.02, 0.04]) if shape == "glm" else 0.0}
    return {"kind": kind, "tokens": _log_int(rng, 1, 4096), "dtype": dtype}


# ---- weights ---------------------------------------------------------------------------------

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _pack(entries):
    """(buffer, meta, views) of a packed layer: ``entries`` = (name, shape, dtype name) in any
    order, laid out by name as the loader does, every tensor aligned."""
    meta, off = [], 0
    for name, shape, dt in sorted(entries):
        off = (off + ALIGN - 1) // ALIGN * ALIGN
        nbytes = math.prod(shape) * ESZ[dt]
        meta.append({"name": name, "shape": list(shape), "dtype": dt, "offset": off,
                     "nbytes": nbytes})
        off += nbytes
    buf = torch.empty(off, dtype=torch.uint8, device="cuda")
    views = {m["name"]: buf[m["offset"]:m["offset"] + m["nbytes"]].view(TORCH[m["dtype"]])
             .view(m["shape"]) for m in meta}
    return buf, meta, views


def _fill(views, name, std, mean, g):
    """N(mean, std) values; int8 matrices are quantised row by row into <name>_scale."""
    v = views[name]
    if v.dtype != torch.int8:
        v.normal_(mean, std, generator=g)
        return
    w = torch.empty(v.shape, dtype=torch.float32, device="cuda").normal_(0, std, generator=g)
    sc = (w.abs().amax(dim=1) / 127).half()
    views[name + "_scale"].copy_(sc)
    v.copy_((w / sc.float()[:, None]).round_().clamp_(-127, 127))


def _with_scales(entries):
    """Adds the fp16 row scales that int8 matrices carry."""
    return entries + [(n + "_scale", [s[0]], "float16") for n, s, d in entries if d == "int8"]


def _norm(views, name, g):
    views[name].normal_(1.0, 0.1, generator=g)


def _moe_entries(shape, dtype):
    return [(m["name"], m["shape"], m["dtype"])
            for m in DeviceMoeLayer.synthetic_meta(shape, dtype, "float32")]


def _fill_moe(shape, views, skew, g):
    for name, _, kind, std in syn.tensor_specs(shape):
        if kind == "norm":
            _norm(views, name, g)
        elif kind == "bias":  # the spread of the correction bias sets how uneven the loads are
            _fill(views, name, math.hypot(std, skew), 0.0, g)
        else:
            _fill(views, name, std, 0.0, g)


def _linear_entries(dtype):
    return _with_scales([(n, list(s), dtype if kind == "weight" else "float32")
                         for n, s, kind, _, _ in syn.linear_attn_specs(LA)])


def _fill_linear(views, g):
    for name, _, kind, std, mean in syn.linear_attn_specs(LA):
        _norm(views, name, g) if kind == "norm" else _fill(views, name, std, mean, g)


def _full_entries(dtype):
    return _with_scales([(n, list(s), dtype if kind == "weight" else "float32")
                         for n, s, kind, _ in syn.full_attn_specs(FA)])


def _fill_full(views, g):
    for name, _, kind, std in syn.full_attn_specs(FA):
        _norm(views, name, g) if kind == "norm" else _fill(views, name, std, 0.0, g)


def _input(tokens, hidden, seed):
    return torch.randn(tokens, hidden, device="cuda", generator=_gen(seed, 17))


def _block_weights(case, seed):
    """(buffer, meta, views) of a single block's weights, row-major."""
    g = _gen(seed)
    if case["kind"] == "moe":
        shape = SHAPES[case["shape"]]
        buf, meta, views = _pack(_moe_entries(shape, case["dtype"]))
        _fill_moe(shape, views, case["skew"], g)
    elif case["kind"] == "linear":
        buf, meta, views = _pack(_linear_entries(case["dtype"]))
        _fill_linear(views, g)
    else:
        buf, meta, views = _pack(_full_entries(case["dtype"]))
        _fill_full(views, g)
    return buf, meta, views


def _stack_weights(case, seed):
    out = []
    for i, kind in enumerate(STACK_KINDS):
        entries = _moe_entries(syn.QWEN3_NEXT, case["dtype"])
        entries += _linear_entries(case["dtype"]) if kind == "linear" else \
            _full_entries(case["dtype"])
        buf, meta, views = _pack(entries)
        g = _gen(seed, 100 + i)
        _fill_moe(syn.QWEN3_NEXT, views, 0.0, g)
        (_fill_linear if kind == "linear" else _fill_full)(views, g)
        out.append((kind, buf, meta, views))
    return out


# ---- the calls -------------------------------------------------------------------------------

def _backend():
    return MI355XBackend(torch.cuda.current_device())


def _stream():
    return torch.cuda.current_stream().cuda_stream or None


class _Block:
    """A block's weights, workspace and buffers, and its call."""

    def __init__(self, case, seed):
        backend, stream = _backend(), _stream()
        T = case["tokens"]
        buf, meta, _ = _block_weights(case, seed)
        base = buf.data_ptr()
        torch.cuda.current_stream().synchronize()
        if case["kind"] == "moe":
            shape = SHAPES[case["shape"]]
            layout = MoeLayerLayout.from_meta(meta)
            tiled = case["layout"] == "frag16"
            if tiled:
                tile_experts(backend, layout, base, stream)
            self.desc = MoeConfig.from_layout(
                layout, top_k=shape.top_k,
                router_mode="sigmoid_select_bias" if shape.has_bias else "softmax",
                norm_topk_prob=True, routed_scaling=shape.routed_scaling, eps=shape.eps,
                weight_layout=_lib.MX_LAYOUT_FRAG16 if tiled else _lib.MX_LAYOUT_ROWS).desc()
            runner = MoeRunner(backend)
            runner.reserve(self.desc, T)
            self.weights = runner.bind(layout, base, stream)
            hidden = shape.hidden
        elif case["kind"] == "linear":
            layout = LinearAttnLayout.from_meta(meta)
            self.desc, self.weights = layout.desc(LA.eps), layout.weights(base)
            runner = LinearAttnRunner(backend)
            runner.reserve(self.desc, T, io=False)
            hidden = LA.hidden
        else:
            layout = FullAttnLayout.from_meta(meta, FA.n_heads, FA.n_kv_heads, FA.head_dim,
                                              FA.rotary_dim, FA.rope_theta)
            self.desc, self.weights = layout.desc(FA.eps), layout.weights(base)
            runner = FullAttnRunner(backend)
            runner.reserve(self.desc, T, io=False)
            hidden = FA.hidden
        self.buf, self.layout, self.runner = buf, layout, runner
        self.x = _input(T, hidden, seed)
        self.out = torch.empty_like(self.x)
        self.tokens = T
        weakref.finalize(self, runner.close)

    def __call__(self):
        self.runner.forward_device(self.desc, self.weights, self.x.data_ptr(),
                                   self.out.data_ptr(), self.tokens, _stream())
        return self.out


def _close_stack(runtime, executor):
    runtime.close()
    executor.close()


class _Stack:
    """Resident layers behind the offload runtime."""

    def __init__(self, case, seed):
        backend = _backend()
        T = case["tokens"]
        specs, buffers, self.keep = [], {}, []
        for i, (kind, buf, meta, _) in enumerate(_stack_weights(case, seed)):
            torch.cuda.current_stream().synchronize()
            tile_experts(backend, MoeLayerLayout.from_meta(meta), buf.data_ptr(), _stream())
            specs.append(make_layer_spec(i, meta, buf.numel(), attn_type=kind,
                                         weight_layout="frag16"))
            buffers[i] = DeviceBuffer(buf.data_ptr(), buf.numel(), backend.name)
            self.keep.append(buf)
        config = {**syn.QWEN3_NEXT.config(), **LA.config(), **FA.config()}
        executor = Qwen3NextExecutor(config, max_tokens=T, device_activations=True)
        self.runtime = OffloadRuntime(specs, backend, DeviceResidentStorage(buffers),
                                      LookaheadScheduler(2), executor, event_timing=False)
        self.ids = [s.layer_id for s in specs]
        self.x = _input(T, FA.hidden, seed).cpu().numpy()
        self.runtime.run_inference(self.ids, self.x)  # the runners' workspaces
        weakref.finalize(self, _close_stack, self.runtime, executor)

    def __call__(self):
        return self.runtime.run_inference(self.ids, self.x)[0]


def prepare(case, seed):
    return _Stack(case, seed) if case["kind"] == "stack" else _Block(case, seed)


def run(state):
    return state()


# ---- what a call cannot do without -----------------------------------------------------------

def _moe_work(shape, dtype, tokens):
    H, E, k, e = shape.hidden, shape.n_experts, shape.top_k, ESZ[dtype]
    active = E * (1.0 - (1.0 - k / E) ** tokens)  # distinct experts of evenly routed tokens
    per = 3 * H * shape.inter * e + (2 * (2 * shape.inter + H) if dtype == "int8" else 0)
    shared = per * shape.shared_inter / shape.inter
    bytes_ = active * per + shared + 4 * E * H + 8 * tokens * H
    flops = 2 * tokens * H * E + 6 * H * tokens * (shape.inter * k + shape.shared_inter)
    return bytes_, flops


def _linear_work(dtype, tokens):
    n, dk, dv, H = LA.n_heads, LA.head_dim_k, LA.head_dim_v, LA.hidden
    w = H * (LA.qkvz_rows + LA.ba_rows + n * dv)
    return w * ESZ[dtype] + 8 * tokens * H, 2 * tokens * w + 5 * tokens * n * dk * dv


def _full_work(dtype, tokens):
    nh, nkv, hd, H = FA.n_heads, FA.n_kv_heads, FA.head_dim, FA.hidden
    w = H * hd * (3 * nh + 2 * nkv)
    return w * ESZ[dtype] + 8 * tokens * H, 2 * tokens * w + 2 * nh * hd * tokens * (tokens + 1)


def work(case):
    T, dt = case["tokens"], case["dtype"]
    if case["kind"] == "moe":
        b, f = _moe_work(SHAPES[case["shape"]], dt, T)
    elif case["kind"] == "linear":
        b, f = _linear_work(dt, T)
    elif case["kind"] == "full":
        b, f = _full_work(dt, T)
    else:
        parts = [_moe_work(syn.QWEN3_NEXT, dt, T)] * 4 + [_linear_work(dt, T)] * 3 + \
            [_full_work(dt, T)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    # Four times the distance from the 64-bit result that was measured: activations are rounded
    # to fp16 before every product (as the package states for fp16 and int8 weights).  A token
    # whose last experts are tied to 32 bits may take either, which "max" leaves room for.
    if case["kind"] == "moe":
        return {"rel": 1.4e-3 if case["shape"] == "glm" else 2.5e-4, "max": 1e-1}
    if case["kind"] == "stack":
        return {"rel": 1.8e-3, "max": 1e-1}
    return {"rel": 1.3e-3 if case["kind"] == "linear" else 8e-4, "max": 5e-2}


# ---- the same in 64 bits ---------------------------------------------------------------------

def _w64(views, name):
    w = views[name].double()
    if views[name].dtype == torch.int8:
        w = w * views[name + "_scale"].double()[:, None]
    return w


def _rms64(x, w, eps):
    r = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)
    return r if w is None else w * r


def _silu(x):
    return x * torch.sigmoid(x)


def _moe64(shape, views, x):
    h = _rms64(x, views["post_attention_layernorm.weight"].double(), shape.eps)
    logits = h @ views["mlp.gate.weight"].double().T
    if shape.has_bias:
        s = torch.sigmoid(logits)
        ids = (s + views["mlp.gate.e_score_correction_bias"].double()).topk(shape.top_k).indices
    else:
        s = torch.softmax(logits, dim=-1)
        ids = s.topk(shape.top_k).indices
    w = s.gather(1, ids)
    w = w / (w.sum(dim=-1, keepdim=True) + 1e-20) * shape.routed_scaling

    def swiglu(a, pre):
        act = _silu(a @ _w64(views, pre + "gate_proj.weight").T) * \
            (a @ _w64(views, pre + "up_proj.weight").T)
        return act @ _w64(views, pre + "down_proj.weight").T

    out = x.clone()
    for e in ids.unique().tolist():
        tok, slot = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, tok, w[tok, slot, None] * swiglu(h[tok], f"mlp.experts.{e}."))
    if shape.shared_inter:
        pre = "mlp.shared_experts." if shape.arch == syn.GLM else "mlp.shared_expert."
        y = swiglu(h, pre)
        if shape.has_shared_gate:
            y = y * torch.sigmoid(h @ views["mlp.shared_expert_gate.weight"].double().T)
        out += y
    return out


def _linear64(views, x):
    n, dk, dv = LA.n_heads, LA.head_dim_k, LA.head_dim_v
    T = x.shape[0]
    h = _rms64(x, views["input_layernorm.weight"].double(), LA.eps)
    qkvz = h @ _w64(views, "linear_attn.in_proj_qkvz.weight").T
    pre, z = qkvz[:, :n * (2 * dk + dv)], qkvz[:, n * (2 * dk + dv):]
    taps = views["linear_attn.conv1d.weight"].double()[:, 0]
    conv = torch.zeros_like(pre)
    for j in range(min(LA.conv_kernel, T)):  # tap 0 weighs the current token
        conv[j:] += pre[:T - j] * taps[:, j]
    q, k, v = _silu(conv).split([n * dk, n * dk, n * dv], dim=1)
    ba = h @ _w64(views, "linear_attn.in_proj_ba.weight").T
    k = (k * torch.sigmoid(ba[:, :n * dk])).view(T, n, dk, 1)
    q, v = q.reshape(T, n, dk, 1), v.reshape(T, n, 1, dv)
    a = ba[:, n * dk:] + views["linear_attn.dt_bias"].double()
    soft = torch.nn.functional.softplus(a, threshold=40.0)
    decay = torch.exp(-views["linear_attn.A_log"].double().exp() * soft).view(T, n, 1, 1)
    state = torch.zeros(n, dk, dv, dtype=torch.float64, device=x.device)
    o = torch.empty(T, n, dv, dtype=torch.float64, device=x.device)
    for t in range(T):
        state = state * decay[t] + k[t] * v[t]
        o[t] = (q[t] * state).sum(dim=1)
    o = _rms64(o.view(T, n * dv), views["linear_attn.norm.weight"].double(), LA.eps) * _silu(z)
    return x + o @ _w64(views, "linear_attn.out_proj.weight").T


def _full64(views, x):
    nh, nkv, hd, rot = FA.n_heads, FA.n_kv_heads, FA.head_dim, FA.rotary_dim
    T = x.shape[0]
    h = _rms64(x, views["input_layernorm.weight"].double(), FA.eps)
    q, gate = (h @ _w64(views, "self_attn.q_proj.weight").T).chunk(2, dim=1)
    k = h @ _w64(views, "self_attn.k_proj.weight").T
    v = (h @ _w64(views, "self_attn.v_proj.weight").T).view(T, nkv, hd)
    # The block defines its RoPE angles as 32-bit numbers, rounded from 64 bits.
    freq = 1.0 / FA.rope_theta ** (torch.arange(rot // 2, dtype=torch.float64) / (rot // 2))
    ang = (torch.arange(T, dtype=torch.float64)[:, None] * freq).float().double().to(x.device)
    c, s = ang.cos()[:, None], ang.sin()[:, None]

    def heads(u, m, norm):
        u = _rms64(u.view(T, m, hd), views[norm].double(), FA.eps)
        a, b = u[..., :rot // 2], u[..., rot // 2:rot]
        return torch.cat([a * c - b * s, b * c + a * s, u[..., rot:]], dim=-1)

    q, k = heads(q, nh, "self_attn.q_norm.weight"), heads(k, nkv, "self_attn.k_norm.weight")
    mask = torch.ones(T, T, dtype=torch.bool, device=x.device).triu(1)
    att = torch.empty(T, nh, hd, dtype=torch.float64, device=x.device)
    for i in range(nh):
        j = i // (nh // nkv)
        p = (q[:, i] @ k[:, j].T / math.sqrt(hd)).masked_fill_(mask, -math.inf)
        att[:, i] = torch.softmax(p, dim=-1) @ v[:, j]
    att = att.view(T, nh * hd) * torch.sigmoid(gate)
    return x + att @ _w64(views, "self_attn.o_proj.weight").T


def exact(case, seed):
    if case["kind"] == "stack":
        x = _input(case["tokens"], FA.hidden, seed).double()
        for kind, _, _, views in _stack_weights(case, seed):
            x = _linear64(views, x) if kind == "linear" else _full64(views, x)
            x = _moe64(syn.QWEN3_NEXT, views, x)
        return x.cpu().numpy()
    _, _, views = _block_weights(case, seed)
    hidden = SHAPES[case["shape"]].hidden if case["kind"] == "moe" else LA.hidden
    x = _input(case["tokens"], hidden, seed).double()
    if case["kind"] == "moe":
        return _moe64(SHAPES[case["shape"]], views, x)
    return _linear64(views, x) if case["kind"] == "linear" else _full64(views, x)
