"""f32 rows of 8192 in registers (up to 1024 rows) and in two passes (past that): the same bits."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,groups", [(8192, 1), (8192, 4), (4104, 1), (6144, 3)])
def test_norm_resadd(H, groups):
    assert ops.native_available(), "HIP extension must be built for GPU tests"
    torch.manual_seed(H)
    y, x, w = torch.randn(1025, H, device="cuda"), torch.randn(1025, H, device="cuda"), torch.randn(H, device="cuda")
    one, lp = x.clone(), torch.empty_like(x)
    seqmix.norm_resadd(y, w, 1e-6, one, lp, groups)
    want = x.double() + torch.nn.functional.normalize(y.double().view(1025, groups, -1), dim=-1).view(1025, H) * (H // groups) ** .5 * w.double()
    assert torch.equal(one, lp) and float((one.double() - want).norm() / want.norm()) < 1e-6
    two = x[:1024].clone()
    seqmix.norm_resadd(y[:1024], w, 1e-6, two, lp[:1024], groups)
    assert torch.equal(one[:1024], two)
