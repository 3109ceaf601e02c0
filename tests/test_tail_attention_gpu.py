"""Attention whose last round of query tiles is partial (kx_attention_tail_fwd): the whole rounds bit-equal
to the plain kernel, the split tiles against it and float64, over partial tiles, several sequences, grouped
heads, gates and ragged keys; and the calls that the rule and the entry point leave out."""

import pytest
import torch

from kinomlx_amd import _lib, workloads
from kinomlx_amd.ltx2.dense_attention import batched_attention

pytestmark = pytest.mark.gpu


def _t(device, shape, seed, dtype):
    return workloads.normal(seed, "tail", shape).to(device, dtype)


def _launch(entry, q, k, v, heads, kv, gate, *more):
    out = torch.full_like(q, float("nan"))
    b, tq, tk = q.shape[0], q.shape[1], k.shape[1]
    sfx = "bf16" if q.dtype == torch.bfloat16 else "f16"
    _lib._call(f"{entry}_{sfx}", q.data_ptr(), q.stride(-2), k.data_ptr(), k.stride(-2), v.data_ptr(), v.stride(-2),
               out.data_ptr(), out.stride(-2), b, tq, tk, heads, kv, 128, 128 ** -0.5,
               None if gate is None else gate.data_ptr(), heads, *more, _lib._stream())
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("batch", "heads", "kv", "tq", "tk", "splits"), [
    (1, 257, 257, 31, 129, 2),     # one tile past the round, its rows partial
    (3, 90, 30, 384, 200, 3),      # 270 tiles, grouped heads, the rest inside the last sequence
    (2, 70, 70, 500, 1000, 4),     # two tiles a head, the second partial
])
def test_tail_slices(device, dtype, batch, heads, kv, tq, tk, splits):
    q, k, v = (_t(device, (batch, n, h * 128), i, dtype) for i, (n, h) in enumerate(((tq, heads), (tk, kv), (tk, kv))))
    gate = _t(device, (batch * tq, heads), 4, dtype)
    tiles = -(-tq // 384)
    blocks = batch * heads * tiles
    full, rest = blocks // 256 * 256, blocks % 256
    work = torch.empty(splits * rest * 384 * 130, dtype=torch.float32, device=device)
    for g in (None, gate):
        got = _launch("kx_attention_tail_fwd", q, k, v, heads, kv, g, work.data_ptr(), work.numel() * 4, splits)
        plain = _launch("kx_attention_gqa_fwd", q, k, v, heads, kv, g)
        a, b = (t.view(batch, tq, heads, 128).transpose(1, 2).reshape(batch * heads, tq, 128).double() for t in (got, plain))
        whole = torch.zeros(batch * heads, tq, dtype=torch.bool, device=device)
        for i in range(full):
            whole[i // tiles, i % tiles * 384:(i % tiles + 1) * 384] = True
        assert torch.equal(a[whole], b[whole])
        qh = q.double().view(batch, tq, heads, 128).transpose(1, 2)
        kh, vh = (t.double().view(batch, tk, kv, 128).transpose(1, 2).repeat_interleave(heads // kv, 1) for t in (k, v))
        s = qh @ kh.transpose(2, 3) * 128 ** -0.5
        p = s.softmax(-1)
        # P rounded to 16 bits (u) in numerator and sum, the output's own rounding, and the fp32 scores
        u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        scale = 1.0 if g is None else g.double().view(batch, tq, heads, 1).transpose(1, 2)
        ref = (p @ vh) * scale
        tol = ((2 * u + 2.0 ** -14) * (p @ vh.abs()) * (1.0 if g is None else scale.abs()) + u * ref.abs() + 2.0 ** -24)
        assert ((a.view(ref.shape) - ref).abs() <= 1.01 * tol).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("batch", "heads", "kv", "tq", "tk"), [
    (1, 3, 3, 1, 257), (2, 4, 2, 256, 300), (1, 4, 4, 257, 1000), (1, 86, 86, 513, 321),  # within one round
    (1, 86, 86, 640, 321)])                                                               # past it: 384-query tiles
def test_small_query_tiles(device, dtype, batch, heads, kv, tq, tk):
    """256-query tiles against the key-sliced form, which keeps 384-query tiles."""
    q, k, v = (_t(device, (batch, n, h * 128), i, dtype) for i, (n, h) in enumerate(((tq, heads), (tk, kv), (tk, kv))))
    gate = _t(device, (batch * tq, heads), 4, dtype)
    got = _launch("kx_attention_gqa_fwd", q, k, v, heads, kv, gate)
    work = torch.empty(2 * batch * heads * tq * 130, dtype=torch.float32, device=device)
    sliced = _launch("kx_attention_split_fwd", q, k, v, heads, kv, gate, None, 0, 0, 0, work.data_ptr(),
                     work.numel() * 4, 2)
    # both round P to 16 bits (u) against their own running max, and the output once
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    size = v.float().abs().amax() * gate.float().abs().view(batch, tq, heads, 1)
    diff = (got.float() - sliced.float()).abs().view(batch, tq, heads, 128)
    assert (diff <= 6 * u * size).all()


def test_rule_and_refusals(device):
    assert _lib.attention_tail(1, 4608, 4608, 32) == 2
    assert _lib.attention_tail(1, 9216, 9216, 32) == 1   # whole rounds
    assert _lib.attention_tail(1, 2628, 2628, 32) == 1   # no whole round
    assert _lib.attention_tail(1, 4608, 512, 32) == 1    # few keys
    q, k = _t(device, (1, 8, 257 * 128), 1, torch.bfloat16), _t(device, (1, 130, 257 * 128), 2, torch.bfloat16)
    work = torch.empty(2 * 384 * 130, dtype=torch.float32, device=device)
    for heads, bytes_, splits in ((256, work.numel() * 4, 2), (255, work.numel() * 4, 2), (257, work.numel() * 4 - 4, 2),
                                  (257, work.numel() * 4, 1)):
        with pytest.raises(_lib.KernelError):
            _launch("kx_attention_tail_fwd", q, k, k, heads, heads, None, work.data_ptr(), bytes_, splits)


def test_both_paths_take_it(device):
    heads, tokens = 32, 4500
    q, k, v = (_t(device, (1, tokens, heads * 128), i, torch.bfloat16) for i in range(3))
    assert _lib.attention_tail(1, tokens, tokens, heads) > 1
    got = batched_attention(q, k, v, heads=heads)
    timer = _lib.LaunchTimer()
    _lib.set_timer(timer)
    try:
        again = batched_attention(q, k, v, heads=heads)
    finally:
        _lib.set_timer(None)
    assert torch.equal(got, again)
    plain = _launch("kx_attention_gqa_fwd", q, k, v, heads, heads, None)
    assert (got.float() - plain.float()).abs().max() <= 2.0 ** -7 * plain.float().abs().max()
