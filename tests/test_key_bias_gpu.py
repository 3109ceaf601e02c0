"""Attention under a mask that is the same for every query (a bias per key, held in LDS): against float64,
over the resident and the streaming form, key slices, both sides of the LDS limit and partial tiles; and
against the general form, which takes the same mask spelled out per query."""

import pytest
import torch

from kinomlx_amd import workloads
from kinomlx_amd.ltx2.dense_attention import batched_attention

pytestmark = pytest.mark.gpu


def _t(device, shape, seed, dtype, std=1.0):
    return workloads.normal(seed, "keybias", shape, std).to(device, dtype)


def _reference(q, k, v, heads, bias, scale):
    """float64 output and its error bound. P is rounded to 16 bits (u) in the numerator and the row sum
    alike: at most 2 u of sum(p |v|); the output's own rounding adds u; the fp32 scores and their bias
    (130 sums and roundings) and exp2 the rest, twice as e^s has slope e^s in numerator and sum."""
    b, tq, tk, d = q.shape[0], q.shape[1], k.shape[1], q.shape[2] // heads
    qh, kh, vh = (t.double().view(b, -1, heads, d).transpose(1, 2) for t in (q, k, v))
    s = qh @ kh.transpose(2, 3) * scale
    bias = bias.double().expand(b, heads, tq, tk)
    removed = bias / scale < -1e20  # -inf and the bf16 minimum; fp16's minimum is a score like others
    all_removed = removed.all(-1, keepdim=True)
    s = torch.where(all_removed, 0.0, torch.where(removed, float("-inf"), s + bias))
    p = s.softmax(-1)
    size = (qh.abs() @ kh.abs().transpose(2, 3) * scale + torch.where(removed, 0.0, bias.abs())).amax(-1, keepdim=True)
    u = 2.0 ** -8 if q.dtype == torch.bfloat16 else 2.0 ** -11
    tol = (2 * u + 2 * (130 * 2.0 ** -24 * size + 2.0 ** -21)) * (p @ vh.abs()) + u * (p @ vh).abs() + 2.0 ** -24
    flat = lambda t: t.transpose(1, 2).reshape(b, tq, heads * d)  # noqa: E731
    return flat(p @ vh), flat(tol) * 1.01


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("tq", "tk"), [(1, 1), (33, 63), (385, 256), (70, 257), (900, 1000), (31, 4096), (5, 4100)])
def test_per_key_masks(device, dtype, tq, tk):
    heads, d, batch, scale = 2, 128, 2, 0.11
    q, k, v = (_t(device, (batch, n, heads * d), i, dtype) for i, n in enumerate((tq, tk, tk)))
    kept = torch.arange(tk, device=device)[None] < torch.tensor([max(1, tk - 29), tk], device=device)[:, None]
    late = torch.zeros(tk, device=device)
    late[:tk - 1] = float("-inf")  # whole tiles removed before the first key that counts
    none = torch.full((tk,), torch.finfo(dtype).min, device=device)
    alibi = -torch.rand((batch, heads, 1, tk), generator=torch.Generator(device).manual_seed(3), device=device) * 20
    for mask in (kept[:, None, None], late.view(1, 1, 1, tk), none.view(1, 1, 1, tk), alibi.to(dtype),
                 torch.stack([late, none]).view(2, 1, 1, tk)):
        bias = torch.where(mask, 0.0, float("-inf")) if mask.dtype == torch.bool else mask
        ref, tol = _reference(q, k, v, heads, bias.to(dtype), scale)
        got = batched_attention(q, k, v, heads=heads, scale=scale, mask=mask)
        assert ((got.double() - ref).abs() <= tol).all()
        general = batched_attention(q, k, v, heads=heads, scale=scale,
                                    mask=bias.to(dtype).expand(-1, -1, tq, -1).contiguous())
        assert ((general.double() - got.double()).abs() <= 2 * tol).all()


def test_large_scores_and_scales(device):
    """Scores far above the 16-bit range beside removed keys, and scales at and past the form's limits."""
    heads, d, tq, tk = 2, 128, 40, 300
    q, k, v = (_t(device, (1, n, heads * d), i, torch.bfloat16, std) for i, (n, std) in
               enumerate(((tq, 200.0), (tk, 200.0), (tk, 1.0))))
    mask = (torch.arange(tk, device=device) % 3 != 0).view(1, 1, 1, tk)
    for scale in (2.0 ** -20, 2.0 ** -21, 1e-3):
        ref, tol = _reference(q, k, v, heads, torch.where(mask, 0.0, float("-inf")), scale)
        got = batched_attention(q, k, v, heads=heads, scale=scale, mask=mask)
        assert ((got.double() - ref).abs() <= tol).all()
