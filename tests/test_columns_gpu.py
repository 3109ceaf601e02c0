"""``kx_gemm_columns_bf16``: the projection whose epilogue normalizes and rotates its query and key
heads (64 or 128 wide) and multiplies out its SwiGLU columns, on every tile it can run on, against the
FP32 oracle; and the layers that take it against their separate passes."""

import numpy as np
import pytest
import torch

import oracle
from kinomlx_amd import _lib, workloads
from kinomlx_amd.flux2.transformer import FeedForward
from kinomlx_amd.kernels import fused_ops
from kinomlx_amd.ltx2.attention import Linear, swiglu_projection
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


def _bf(shape, seed, std=1.0):
    return workloads.bf16(workloads.normal(seed, "columns", shape, std))


def _np(t):
    return t.float().cpu().numpy()


@pytest.mark.parametrize("tile", ["auto", "0", "1", "2", "3"])
@pytest.mark.parametrize(
    ("m", "k", "head_dim", "heads", "v_width", "ff", "bias"),
    [(300, 128, 64, 2, 128, 0, True),      # heads only, 64 wide, ragged rows
     (70, 192, 64, 4, 256, 384, False),    # 64-wide heads, V, SwiGLU
     (257, 128, 128, 2, 256, 256, True),   # one row past a tile
     (129, 64, 128, 0, 0, 640, True)])     # SwiGLU only
def test_columns_match_the_oracle(device, monkeypatch, tile, m, k, head_dim, heads, v_width, ff, bias):
    if tile != "auto":
        monkeypatch.setenv("KX355_GEMM_LDS_TILE", tile)
    width = heads * head_dim
    begin = 2 * width + v_width
    n = begin + 2 * ff
    x, w, b = _bf((m, k), 1), _bf((n, k), 2, 0.1), _bf((n,), 3, 0.5)
    nq, nk = workloads.normal(4, "nq", (head_dim,), 0.2, 1.0), workloads.normal(5, "nk", (head_dim,), 0.2, 1.0)
    angle = workloads.normal(6, "angle", (m, head_dim // 2), 2.0).repeat_interleave(2, dim=-1)
    cos, sin = angle.cos(), angle.sin()
    out = torch.full((m, begin + 8), 7.0, dtype=torch.bfloat16, device=device)
    joined = torch.full((m, ff + 16), 7.0, dtype=torch.bfloat16, device=device)
    args = {}
    if heads:
        args = dict(q_end=width, k_end=2 * width, head_dim=head_dim, norm_q=nq.to(device), norm_k=nk.to(device),
                    eps=1e-6, cos=cos.to(device), sin=sin.to(device), table_ld=head_dim, table_rows=m)
    if ff:
        args.update(swiglu_begin=begin, swiglu_out=joined[:, 8:8 + ff])
    _lib.launch_gemm_columns(x.to(device), w.to(device), out[:, :begin] if begin else None,
                             bias=b.to(device) if bias else None, **args)
    lin = oracle.linear(_np(x), _np(w), _np(b) if bias else None)
    got = _np(out)
    assert np.all(got[:, begin:] == 7.0)
    if heads:
        raw = oracle.to_bf16(lin[:, :2 * width])
        for lo, weight in ((0, nq), (width, nk)):
            h = oracle.rms_norm(raw[:, lo:lo + width].reshape(m, heads, head_dim), weight.numpy(), 1e-6)
            ref = oracle.pair_rope(h, cos.numpy()[:, None], sin.numpy()[:, None]).reshape(m, width)
            # one rounding of the result, and the projection's own rounding of either pair member
            assert rel_l2(got[:, lo:lo + width], ref) < 4e-3
    plain = lin[:, 2 * width:begin]
    assert np.all(np.abs(got[:, 2 * width:begin] - plain) <= np.abs(plain) * 2.0**-7 + 1e-4 * np.abs(lin).max())
    if ff:
        sw = _np(joined)
        assert np.all(sw[:, :8] == 7.0) and np.all(sw[:, 8 + ff:] == 7.0)
        gate, up = lin[:, begin:begin + ff], lin[:, begin + ff:]
        ref = oracle.silu(gate) * up
        # one bf16 rounding, the products' summation order, and the fast exp / reciprocal of silu
        assert np.all(np.abs(sw[:, 8:8 + ff] - ref) <= np.abs(ref) * 2.0**-7 + 2e-4 * np.abs(lin).max() * (1 + np.abs(up)))


def test_feed_forward_with_and_without_the_fused_swiglu_agree(device):
    """The fused layer rounds once where the separate passes round gate, up and product: no further
    from FP32 than they are. Layers outside the contract keep the passes."""
    layer = FeedForward()
    layer.linear_in, layer.linear_out = Linear(_bf((512, 256), 7, 0.1).to(device)), Linear(_bf((256, 256), 8, 0.1).to(device))
    x = _bf((2, 75, 256), 9).to(device)
    fused = swiglu_projection(layer.linear_in, x)
    passes = fused_ops.swiglu(layer.linear_in(x))
    lin = x.float() @ layer.linear_in.weight.float().t()
    ref = torch.nn.functional.silu(lin[..., :256]) * lin[..., 256:]
    assert fused.shape == passes.shape == (2, 75, 256)
    assert rel_l2(_np(fused), _np(ref)) <= rel_l2(_np(passes), _np(ref)) < 4e-3
    # six independent bf16 roundings lie between the two outputs (product, gate, up and product again,
    # and each output), at most 2^-9 RMS each: sqrt(6) 2^-9 = 4.8e-3
    assert rel_l2(_np(layer(x)), _np(layer.linear_out(passes))) < 4.8e-3
    odd = Linear(_bf((384, 256), 10, 0.1).to(device))  # 192 gate columns: not whole tiles
    assert swiglu_projection(odd, x) is None
    assert swiglu_projection(layer.linear_in, x.half()) is None
