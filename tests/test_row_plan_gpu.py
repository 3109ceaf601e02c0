"""The dense products' row split (whole rounds of 256 x 256 tiles, then the remaining rows on a smaller
tile): bit-identical to one tile size over all rows (every tile sums K in the same order), for every
epilogue that counts rows from the product's first one."""

import pytest
import torch

from kinomlx_amd import _lib, workloads
from kinomlx_amd.kernels.mpp_linear import fused_linear

M, N, K = 1111, 16384, 1024  # 320 tiles of 256 x 256: one whole round, then 87 rows


def _bf(shape, seed, std=1.0):
    return workloads.bf16(workloads.normal(seed, "rows", shape, std))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("epi", ["bias_gelu", "gated_f32", "gated_rows", "gated_half"])
def test_row_split_equals_one_tile_size(device, monkeypatch, epi, dtype):
    x, w, b = (_bf(s, i, std).to(device, dtype) for i, (s, std) in enumerate((((M, K), 1.0), ((N, K), 0.02), ((N,), 0.1))))
    kwargs = {}
    if epi == "bias_gelu":
        kwargs = dict(activation="gelu_tanh")
    else:
        resid = workloads.normal(3, "resid", (M, N)).to(device)
        gate = workloads.normal(4, "gate", (M, N) if epi == "gated_rows" else (N,), 0.5).to(device)
        kwargs = dict(residual=resid.to(dtype) if epi == "gated_half" else resid, gate=gate, out_dtype=torch.float32)
    split = fused_linear(x, w, b, **kwargs)
    monkeypatch.setenv("KX355_GEMM_LDS_TILE", "0")
    assert torch.equal(split, fused_linear(x, w, b, **kwargs))


@pytest.mark.gpu
def test_row_split_of_the_norm_rope_projection_reads_its_own_table_rows(device, monkeypatch):
    """Two sequences of tables: the split part's rows index them from the product's first row."""
    rows, tokens = 2 * 556, 556
    x, w = _bf((rows, K), 5).to(device), _bf((N, K), 6, 0.02).to(device)
    nq = torch.ones(128, device=device)
    angle = workloads.normal(7, "angle", (2, tokens, 128)).to(device)
    cos, sin = angle.cos().contiguous(), angle.sin().contiguous()

    def call():
        out = torch.empty((rows, N), dtype=torch.bfloat16, device=device)
        _lib.launch_gemm_qknorm_rope(x, w, out, bias=None, q_end=4096, k_end=8192, norm_q=nq, norm_k=nq, eps=1e-6,
                                     weight_offset=0.0, cos=cos, sin=sin, table_ld=128, table_hs=0,
                                     table_rows=tokens, table_bs=tokens * 128)
        return out

    split = call()
    monkeypatch.setenv("KX355_GEMM_LDS_TILE", "0")
    assert torch.equal(split, call())


def test_split_rule_is_a_pure_function_of_the_sizes():
    for m, n, k in [(480, 4096, 16384), (1111, 4096, 16384), (5, 4096, 4096)]:
        s = _lib.splitk_splits(m, n, k)
        assert s > 1 and k % (64 * s) == 0 and k // s >= 256
    assert _lib.splitk_splits(4608, 512, 8192) == 1  # few columns, many rows: one summation order
    assert _lib.splitk_splits(1111, 16384, 4096) == 1
    assert _lib.splitk_splits(4, 4096, 16384) == 1  # the few-row kernel
    with pytest.raises(_lib.KernelError):
        _lib.splitk_splits(1 << 31, 4096, 4096)
