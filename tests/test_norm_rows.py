"""Rows of at most 512 without a residual, a wave a row, against the form with one (a residual of zeros): equal bits."""
import pytest
import torch

from distributed_llm_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 4, 5, 130])
@pytest.mark.parametrize("H", [8, 64, 504, 512, 520])
@pytest.mark.parametrize("layernorm", [False, True])
def test_against_the_form_with_a_residual(rows, H, layernorm):
    torch.manual_seed(rows + H)
    x = (torch.randn(rows, H + 16, device="cuda") * 3).to(torch.bfloat16)[:, 8:H + 8]
    w, b = ((torch.randn(H, device="cuda") + k).to(torch.bfloat16) for k in (1, 0))
    x[rows // 2, H // 2] = float("nan")
    x[0, 0] = float("inf")
    f = (lambda **r: ops.layer_norm(x, w, b, 1e-5, **r)) if layernorm else (lambda **r: ops.rms_norm(x, w, 1e-5, **r))
    got, want = f(), f(residual=torch.zeros(rows, H, device="cuda", dtype=torch.bfloat16))
    assert got[1:].isfinite().any() or rows < 3
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
