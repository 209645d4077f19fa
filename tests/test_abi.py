"""The C-ABI library loads and exports every entry point include/moe_mi355x.h declares;
host-side argument validation (no GPU work) behaves as documented."""
from __future__ import annotations

import ctypes
import re
from pathlib import Path

import pytest

from moe_mi355x import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "moe_mi355x.h"


def declared_functions() -> list[str]:
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(mx_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_abi():
    names = declared_functions()
    assert "mx_moe_forward" in names and "mx_malloc" in names and len(names) >= 30


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, f"symbols declared but not exported: {missing}"


def test_bindings_cover_the_header():
    assert set(declared_functions()) == set(_lib.exported_names())


def _desc(**kw):
    d = dict(hidden=64, inter=32, shared_inter=32, n_experts=8, top_k=2, router_mode=0,
             norm_topk_prob=1, weight_dtype=_lib.MX_DT_F16, param_dtype=_lib.MX_DT_F32,
             has_bias=1, has_shared_gate=0, routed_scaling=2.5, eps=1e-5)
    d.update(kw)
    return _lib.MxMoeDesc(**d)


def _ws(desc, T):
    n = ctypes.c_size_t()
    rc = _lib.load().mx_moe_workspace_size(ctypes.byref(desc), T, ctypes.byref(n))
    return rc, n.value


def test_workspace_size_grows_with_tokens():
    d = _desc()
    rc1, n1 = _ws(d, 1)
    rc2, n2 = _ws(d, 4096)
    assert rc1 == rc2 == _lib.MX_OK and 0 < n1 < n2


@pytest.mark.parametrize("wdt", [_lib.MX_DT_F32, _lib.MX_DT_F16, _lib.MX_DT_I8])
@pytest.mark.parametrize("shape", [
    dict(hidden=5120, inter=1536, shared_inter=1536, n_experts=160, top_k=8),
    dict(hidden=2048, inter=512, shared_inter=512, n_experts=512, top_k=10, has_bias=0,
         has_shared_gate=1),
    dict(hidden=512, inter=32, shared_inter=0, n_experts=8, top_k=1, param_dtype=_lib.MX_DT_F16),
    dict(hidden=64, inter=32, shared_inter=0, n_experts=1024, top_k=1)])
def test_moe_workspace_never_shrinks_with_tokens(wdt, shape):
    """A workspace sized for a batch serves every shorter one (the runners size it once), although
    the router's slices and the m-tile lists get fewer as tokens grow."""
    d = _desc(weight_dtype=wdt, **shape)
    edge = 2 ** 31 // (4 * d.hidden)  # the router's GEMMs end at 2 GiB of activations
    tokens = [*range(0, 2100), *range(2100, 4200, 37), *range(4200, 300000, 20011),
              131071, 131072, 131073, *sorted({edge - 1, edge, edge + 1, 2 * edge - 1, 2 * edge, 2 * edge + 1})]
    sizes = [_ws(d, T)[1] for T in sorted(tokens)]
    assert sizes == sorted(sizes)


@pytest.mark.parametrize("wdt,hidden,inter,E,k,shared,T,m_blk", [
    (_lib.MX_DT_I8, 5120, 1536, 160, 8, 1536, 160, 16),   # 8 rows per expert
    (_lib.MX_DT_I8, 5120, 1536, 160, 8, 1536, 161, 32),
    (_lib.MX_DT_I8, 5120, 1536, 160, 8, 1536, 320, 32),   # 16 rows, experts past 4 MiB
    (_lib.MX_DT_I8, 5120, 1536, 160, 8, 1536, 321, 128),
    (_lib.MX_DT_I8, 2048, 1024, 128, 8, 1024, 384, 32),   # 24 rows, experts of 4 MiB
    (_lib.MX_DT_I8, 2048, 1024, 128, 8, 1024, 385, 128),
    (_lib.MX_DT_I8, 2048, 1040, 128, 8, 1040, 257, 128),  # just past them
    (_lib.MX_DT_I8, 5120, 1536, 16, 6, 1536, 64, 32),     # 24 rows up to 64 tokens
    (_lib.MX_DT_I8, 5120, 1536, 15, 6, 1536, 64, 64),
    (_lib.MX_DT_F16, 2048, 512, 512, 10, 512, 102, 32),   # 2 rows
    (_lib.MX_DT_F16, 2048, 512, 512, 10, 512, 103, 128),
    (_lib.MX_DT_F16, 2048, 512, 64, 2, 1024, 96, 32),     # 3 rows with a heavy shared expert
    (_lib.MX_DT_F16, 2048, 512, 64, 2, 1023, 96, 128),
    (_lib.MX_DT_F16, 2048, 512, 1024, 1, 512, 128, 16),
    (_lib.MX_DT_F16, 2048, 512, 1024, 1, 512, 129, 128),
    (_lib.MX_DT_F32, 2048, 512, 512, 10, 512, 65, 64)])
def test_rows_per_tile(wdt, hidden, inter, E, k, shared, T, m_blk):
    """Both sides of each line of the tile-height rule, read from the workspace views."""
    d = _desc(weight_dtype=wdt, hidden=hidden, inter=inter, n_experts=E, top_k=k,
              shared_inter=shared)
    v = _lib.MxMoeViews()
    rc = _lib.load().mx_moe_views(ctypes.byref(d), T, ctypes.c_void_p(1 << 12), ctypes.byref(v))
    assert rc == _lib.MX_OK and v.m_blk == m_blk


@pytest.mark.parametrize("field,value", [("top_k", 0), ("top_k", 9), ("router_mode", 3),
                                         ("weight_dtype", 7), ("param_dtype", 2),
                                         ("hidden", 0), ("n_experts", -1)])
def test_bad_descriptor_is_rejected(field, value):
    rc, _ = _ws(_desc(**{field: value}), 8)
    assert rc == _lib.MX_ERR_INVALID


def test_shared_gate_needs_shared_expert():
    rc, _ = _ws(_desc(shared_inter=0, has_shared_gate=1), 8)
    assert rc == _lib.MX_ERR_INVALID


def test_null_pointers_rejected_before_any_launch():
    lib = _lib.load()
    assert lib.mx_rmsnorm(None, None, 0, 1e-5, 4, 64, None, None, None) == _lib.MX_ERR_INVALID
    assert lib.mx_combine(None, None, None, 4, 64, 2, 0, None, None) == _lib.MX_ERR_INVALID
    assert lib.mx_malloc(None, 16) == _lib.MX_ERR_INVALID
    d = _desc()
    w = _lib.MxMoeWeights()
    assert lib.mx_moe_forward(ctypes.byref(d), ctypes.byref(w), None, None, 4, None, 0,
                              None) == _lib.MX_ERR_INVALID


def test_error_strings():
    assert _lib.error_string(_lib.MX_ERR_WORKSPACE) == "workspace too small"
    with pytest.raises(ValueError):
        _lib.check(_lib.MX_ERR_INVALID, "x")
    with pytest.raises(RuntimeError):
        _lib.check(_lib.MX_ERR_UNSUPPORTED, "x")


def test_noalloc_refuses_batches_beyond_its_scratch_on_the_host():
    """mx_moe_forward_noalloc checks the batch's workspace against its fixed scratch before
    any HIP call: an oversized batch or a bad descriptor is refused here, without a GPU."""
    lib = _lib.load()
    w = _lib.MxMoeWeights()
    big = _desc(hidden=5120, inter=1536, shared_inter=1536, n_experts=160, top_k=8)
    T = 1
    while _ws(big, T)[1] <= _lib.MX_NOALLOC_MAX_WORKSPACE:
        T *= 2
    assert lib.mx_moe_forward_noalloc(ctypes.byref(big), ctypes.byref(w), None, None, T,
                                      None) == _lib.MX_ERR_WORKSPACE
    assert lib.mx_moe_forward_noalloc(ctypes.byref(_desc(top_k=0)), ctypes.byref(w), None,
                                      None, 4, None) == _lib.MX_ERR_INVALID
