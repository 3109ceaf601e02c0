"""Dense products of 1 to 4 rows (and 5, the first on the tiles) against float64: K below, at and past the
512-wide pieces and the four waves' shares of them, columns off the groups of four, every epilogue, strided
rows, and infinities and NaN kept to their own row."""

import pytest
import torch

from kinomlx_amd import workloads
from kinomlx_amd.kernels.mpp_linear import fused_linear

pytestmark = pytest.mark.gpu


def _t(device, shape, seed, dtype, std=1.0):
    return workloads.normal(seed, "fewrows", shape, std).to(device, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5])
@pytest.mark.parametrize(("n", "k"), [(4, 8), (37, 512), (130, 520), (256, 2048), (68, 2056), (1024, 4096), (5, 8200)])
def test_few_rows_match_float64(device, dtype, m, n, k):
    x = _t(device, (m, k + 8), 1, dtype)[:, :k]
    w, b = _t(device, (n, k + 16), 2, dtype, 0.05)[:, :k], _t(device, (n,), 3, dtype)
    resid, gate = _t(device, (m, n), 4, torch.float32), _t(device, (n,), 5, torch.float32)
    exact = x.double() @ w.double().t()
    # fp32 sums of k products: k * 2^-24 of the sum of the magnitudes (2 more roundings for the epilogue), and
    # the output's own rounding: 2^-8 of it with bf16's 8 significant bits, 2^-11 with fp16's 11
    size = x.double().abs() @ w.double().abs().t()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    tol = (k + 2) * 2.0 ** -24 * (size + b.double().abs())
    def check(got, ref, tol):
        half = unit * 1.01 * ref.abs() if got.dtype == dtype else 2.0 ** -23 * ref.abs()
        assert ((got.double() - ref).abs() <= tol + half + 2.0 ** -24).all()

    out = dtype if n % 4 else torch.float32  # fp32 rows are 16-byte aligned
    check(fused_linear(x, w), exact, tol)
    check(fused_linear(x, w, b, out_dtype=out), exact + b.double(), tol)
    ref = resid.to(out).double() + gate.double() * exact
    check(fused_linear(x, w, residual=resid.to(out), gate=gate, out_dtype=out), ref, tol * gate.double().abs())


def test_non_finite_values_stay_in_their_row(device):
    x, w = _t(device, (3, 1032), 6, torch.bfloat16), _t(device, (64, 1032), 7, torch.bfloat16)
    clean = fused_linear(x, w)
    x[1, 1031] = float("inf")
    x[2, 0] = float("nan")
    got = fused_linear(x, w)
    assert torch.equal(got[0], clean[0]) and got[1].isinf().all() and got[2].isnan().all()
