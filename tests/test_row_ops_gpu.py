"""Row passes at the edges of their vector forms: register-row AdaLN widths, split RoPE on 64-wide
heads (one tensor, and Q with K), 16-byte against element-wise accesses, and Krea 2's folded
modulation rows."""

import numpy as np
import pytest
import torch

import oracle
from kinomlx_amd import _lib, workloads
from kinomlx_amd.kernels import fused_ops
from kinomlx_amd.krea2.transformer import split_six_way_modulation
from kinomlx_amd.ltx2.attention import RMSNorm, norm_rope, norm_rope_qk
from kinomlx_amd.ltx2.transformer import adaln, gated_residual, layer_norm_modulate, modulate
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu
ULP = 2.0**-7  # bf16


def _t(shape, seed, std=1.0, mean=0.0):
    return workloads.normal(seed, "rowops", shape, std, mean)


def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim", [512, 1536, 2560, 3072, 3584, 4608, 5120, 6144])
def test_adaln_widths(device, dim, dtype, kind):
    """3584 and 4608 (seven and nine vectors) keep the strided loop."""
    x = _t((1, 5, dim), dim).to(dtype)
    scale, shift = _t((1, 1, dim), 1), _t((1, 1, dim), 2)
    fn, ref = {
        "rms": (lambda: adaln(x.to(device), scale.to(device), shift.to(device), 1e-6), oracle.rms_norm(x.float().numpy())),
        "layer": (lambda: layer_norm_modulate(x.to(device), shift.to(device), scale.to(device)),
                  oracle.layer_norm(x.float().numpy())),
    }[kind]
    ref = ref * (1 + scale.numpy()) + shift.numpy()
    assert np.all(np.abs(_np(fn()) - ref) <= np.abs(ref) * ULP + 1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dim", [1024, 2048, 4096])
@pytest.mark.parametrize("offset", [0, 1])
def test_split_rope_of_64_wide_heads(device, dim, dtype, offset):
    """Norm + RoPE of one tensor against the oracle, with an aligned weight and one that
    starts an element later; Q and K in one pass give the same bits as one at a time."""
    heads, tokens = dim // 64, 7
    q, k = (_t((2, tokens, dim), s).to(device, dtype) for s in (1, 2))
    weights = [_t((dim + offset,), s, 0.1, 1.0).to(device, dtype)[offset:] for s in (3, 4)]
    angle = _t((1, tokens, heads, 32), 5, 2.0)
    pe = tuple(f(angle).to(device).transpose(1, 2) for f in (torch.cos, torch.sin))
    norms = [RMSNorm(dim, weight=w) for w in weights]
    one = [norm_rope(x, n, pe, heads) for x, n in zip((q, k), norms)]
    both = norm_rope_qk(q, k, *norms, pe, heads)
    assert all(torch.equal(a, b) for a, b in zip(one, both))
    for x, n, got in zip((q, k), norms, one):
        normed = oracle.rms_norm(_np(x), _np(n.weight))
        ref = oracle.split_rope(normed, _np(pe[0]), _np(pe[1]))
        # one rounding of the 16-bit result
        assert rel_l2(_np(got), ref) < (2.5e-3 if dtype == torch.bfloat16 else 3.2e-4)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_vector_and_element_accesses_agree(device, dtype):
    """The same rows at a 16-byte aligned address and one element later."""
    rows, dim = 3, 264
    base = _t((rows, 2 * dim + 8), 6).to(device, dtype)
    shift, scale = _t((1, dim), 7).to(device), _t((1, dim), 8).to(device)
    moved = torch.empty((rows, 2 * dim + 9), dtype=dtype, device=device)[:, 1:]
    moved.copy_(base)
    for fn in (lambda x: modulate(x[:, :dim], scale, shift), lambda x: gated_residual(x[:, :dim], x[:, dim:2 * dim], scale)):
        assert torch.equal(fn(base), fn(moved))
    out = torch.empty((rows, dim), dtype=dtype, device=device)
    odd = torch.empty((rows, dim + 1), dtype=dtype, device=device)[:, 1:]
    _lib.launch_swiglu(base[:, :2 * dim], out)
    _lib.launch_swiglu(base[:, :2 * dim], odd)
    assert torch.equal(out, odd) and torch.equal(out, fused_ops.swiglu(base[:, :2 * dim].contiguous()))


@pytest.mark.parametrize("shape", [(1,), (3,), (2, 5)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_six_way_modulation_folds_the_norm_weights(device, shape, dtype):
    dim = 136
    projected = _t((*shape, 6 * dim), 9).to(device, dtype)
    table, w1, w2 = _t((6, dim), 10).to(device), _t((dim,), 11, 0.3).to(device), _t((dim,), 12, 0.3).to(device)
    rows = list(split_six_way_modulation(projected.float(), table))
    rows[0] = (1.0 + rows[0]) * (1.0 + w1) - 1.0
    rows[3] = (1.0 + rows[3]) * (1.0 + w2) - 1.0
    got = _lib.six_way_modulation(projected, table, w1, w2)
    assert got.shape == (*shape, 6, dim) and got.dtype == torch.float32
    assert torch.equal(got, torch.stack(rows, dim=-2))
