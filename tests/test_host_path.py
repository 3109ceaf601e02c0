"""The native launch path (``csrc/host.cpp``) against the Python path behind it: the same bits for every
layout, type and option that either takes, the same refusals, and CPU tensors left to Python. A
``LaunchTimer`` keeps calls on the Python path."""

import contextlib

import pytest
import torch

from kinomlx_amd import _lib, workloads
from kinomlx_amd.kernels.mpp_linear import fused_linear
from kinomlx_amd.ltx2.attention import RMSNorm, norm_rope, norm_rope_qk
from kinomlx_amd.ltx2.dense_attention import batched_attention
from kinomlx_amd.ltx2.transformer import adaln, layer_norm_modulate, modulate


@contextlib.contextmanager
def python_path():
    _lib.set_timer(_lib.LaunchTimer())
    try:
        yield
    finally:
        _lib.set_timer(None)


def _t(device, shape, seed, dtype=torch.bfloat16, std=1.0):
    return workloads.normal(seed, "host", shape, std).to(device, dtype)


def _agree(fn):
    """``fn()`` on both paths: equal tensors, or the same exception type and text."""
    results = []
    for path in (contextlib.nullcontext, python_path):
        with path():
            try:
                got = fn()
                results.append(got if isinstance(got, tuple) else (got,))
            except (ValueError, RuntimeError, ZeroDivisionError) as exc:
                results.append((type(exc), str(exc).split("(")[0]))
    a, b = results
    assert len(a) == len(b)
    for x, y in zip(a, b):
        if isinstance(x, torch.Tensor):
            assert isinstance(y, torch.Tensor) and x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)
        else:
            assert x == y
    return a


def test_cpu_tensors_and_other_objects_are_left_to_python():
    native = _lib._bind_host()
    x, w = torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(8, 64, dtype=torch.bfloat16)
    assert native.linear(x, w, None, 0, None, None, None, -1, 0) is None
    assert native.linear(None, w, None, 0, None, None, None, -1, 0) is None
    assert native.attention(x, x, x, 0, 0, None, None, None, 0) is None
    assert native.norm(x, w, 1e-6, None, None, 0, 0) is None
    assert native.table_add(x, None, 0, 0) is None
    with pytest.raises(TypeError):
        native.linear(x, w)
    with python_path():
        assert _lib.host() is None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_linear(device, dtype):
    m, n, k = 37, 136, 192
    x, w, b = _t(device, (2, m, k), 1, dtype), _t(device, (n, k), 2, dtype, 0.1), _t(device, (n,), 3, dtype)
    resid, gate = _t(device, (2, m, n), 4, torch.float32), _t(device, (1, 1, n), 5, torch.float32)
    wide = _t(device, (2, m, k + 64), 6, dtype)
    odd = _t(device, (2, m, k + 4), 7, dtype)
    _agree(lambda: fused_linear(x, w, b))
    _agree(lambda: fused_linear(x, w, None, activation="gelu_tanh"))
    _agree(lambda: fused_linear(x, w, b, out_dtype=torch.float32))
    _agree(lambda: fused_linear(wide[..., :k], w, b))          # a column slice
    _agree(lambda: fused_linear(odd[..., 4:], w, b))           # rows that need a copy
    _agree(lambda: fused_linear(x.transpose(0, 1), w, b))      # leading axes that do not flatten
    _agree(lambda: fused_linear(x, w.t().contiguous().t(), b))  # a weight that needs a copy
    _agree(lambda: fused_linear(x[0, 0], w, b))                # one row
    _agree(lambda: fused_linear(x[:, :0], w, b))               # none
    for g in (gate, gate[0, 0], _t(device, (2, 1, n), 8, torch.float32), _t(device, (2, m, n), 9, torch.float32),
              gate.to(dtype)):
        _agree(lambda: fused_linear(x, w, b, residual=resid, gate=g, out_dtype=torch.float32))
        _agree(lambda: fused_linear(x, w, b, residual=resid.to(dtype), gate=g))
    buffer = torch.zeros((2 * m, n + 8), dtype=dtype, device=device)
    got = fused_linear(x[0], w, b, out=buffer[:m, :n])
    assert got.data_ptr() == buffer.data_ptr() and not buffer[m:].any() and not buffer[:, n:].any()
    assert torch.equal(got, fused_linear(x[0], w, b))
    for bad in (lambda: fused_linear(x.float(), w, b), lambda: fused_linear(x, w[:, :k - 8].contiguous(), b),
                lambda: fused_linear(x, w, b[:-1]), lambda: fused_linear(x, w, b.float()),
                lambda: fused_linear(x, w, b, residual=resid), lambda: fused_linear(x, w.float(), b)):
        assert _agree(bad)[0] is ValueError
    # K slices and the tail split, by the same plan on both paths
    for m, n, k in ((127, 2048, 2048), (4352, 4096, 8192)):
        x, w = _t(device, (m, k), 10, dtype), _t(device, (n, k), 11, dtype, 0.02)
        _agree(lambda: fused_linear(x, w))
    rows = _t(device, (m, n), 12, torch.float32)  # a gate per row keeps the one plain launch
    _agree(lambda: fused_linear(x, w, residual=rows, gate=rows, out_dtype=torch.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_passes(device, dtype):
    x = _t(device, (2, 9, 1024), 1, dtype)
    for shape in ((1024,), (1, 1, 1024), (2, 1, 1024), (2, 9, 1024)):
        scale, shift = _t(device, shape, 2, torch.float32), _t(device, shape, 3, torch.float32)
        for fn in (lambda v: adaln(v, scale, shift, 1e-6), lambda v: layer_norm_modulate(v, shift, scale),
                   lambda v: modulate(v, scale, shift)):
            _agree(lambda: fn(x))
            _agree(lambda: fn(x[:, ::2]))
            _agree(lambda: fn(x[..., 1:]))
    _agree(lambda: adaln(x.float(), scale, shift, 1e-6, dtype))
    _agree(lambda: adaln(x.float(), scale[:, :1], shift, 1e-6))
    _agree(lambda: adaln(x, scale.to(dtype), shift, 1e-6))
    assert _agree(lambda: adaln(x, scale, shift, 1e-6, torch.float32))[0] is ValueError
    assert _agree(lambda: adaln(x.double(), scale, shift, 1e-6))[0] is ValueError
    table, ts = _t(device, (9, 64), 4, torch.float32), _t(device, (2, 3, 9, 64), 5, dtype)
    _agree(lambda: _lib.table_add(table[2:4], ts[:, :, 2:4]))
    _agree(lambda: _lib.table_add(table, ts[:, :1, :, :].expand(-1, 3, -1, -1), round_to=dtype))
    _agree(lambda: _lib.table_add(table, None))
    assert _agree(lambda: _lib.table_add(table, ts[..., :32]))[0] is ValueError


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim", [64, 128, 32])
def test_norms(device, head_dim):
    batch, tokens, dim = 2, 5, 1024
    heads = dim // head_dim
    qkv = _t(device, (batch, tokens, 2 * dim), 1)
    q, k = qkv[..., :dim], qkv[..., dim:]
    norms = [RMSNorm(dim, weight=_t(device, (dim,), s, dt)) for s, dt in ((2, torch.bfloat16), (3, torch.float32))]
    for tables in (1, batch):
        angle = _t(device, (tables, tokens, heads, head_dim // 2), 4, torch.float32)
        pe = (angle.cos().transpose(1, 2), angle.sin().transpose(1, 2))
        headed = tuple(t.contiguous() for t in pe)  # head-major storage: laid out again by Python
        for p in (None, pe, headed):
            for norm in norms:
                _agree(lambda: norm_rope(q, norm, p, heads))
        for p in (pe, headed):
            pair = [norms[0], RMSNorm(dim, weight=norms[0].weight * 2)]
            if head_dim != 32:
                _agree(lambda: norm_rope_qk(q, k, *pair, p, heads))
        assert _agree(lambda: norm_rope(q, norms[0], (pe[0][:, :, 1:], pe[1][:, :, 1:]), heads))[0] is ValueError


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("tq", "tk", "dim", "kv"), [(33, 70, 128, 4), (50, 1100, 64, 2), (5, 5, 64, 4)])
def test_attention(device, dtype, tq, tk, dim, kv):
    heads, batch = 4, 2
    q = _t(device, (batch, tq, 3 * heads * dim), 1, dtype)[..., :heads * dim]
    keys = _t(device, (batch, tk, 2 * kv * dim), 2, dtype)
    k, v = keys[..., :kv * dim], keys[..., kv * dim:]
    gate = _t(device, (batch, tq, heads), 3, dtype)
    groups = None if kv == heads else kv
    _agree(lambda: batched_attention(q, k, v, heads=heads, kv_heads=groups))
    _agree(lambda: batched_attention(q, k, v, heads=heads, kv_heads=groups, gate=gate, scale=0.2))
    _agree(lambda: batched_attention(q[:1], k[:1], v[:1], heads=heads, kv_heads=groups, gate=gate[:1]))
    for bad in (dict(heads=3), dict(heads=heads, kv_heads=3), dict(heads=4096), dict(heads=heads, gate=gate.float())):
        assert _agree(lambda: batched_attention(q, k, v, **{"kv_heads": groups, **bad}))[0] is ValueError
