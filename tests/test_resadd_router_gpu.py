"""norm_resadd and the router of its rounded rows in one launch (resadd_router_kernel, csrc/kernels/elementwise.hip): the bits of the two launches."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T", [1, 5, 300, 2049])
@pytest.mark.parametrize("H", [8, 504, 512, 520, 1024, 1032, 2048, 2056])
@pytest.mark.parametrize("E,k,shared", [(1, 1, False), (7, 2, True), (8, 2, True), (9, 8, False), (64, 6, True)])
def test_the_two_launches(T, H, E, k, shared):
    torch.manual_seed(T + H + E)
    y = torch.randn(T, H + 3, device=DEV).bfloat16()[:, :H]
    w, bias = torch.randn(H, device=DEV), torch.randn(H, device=DEV) if E != 8 else None
    wg = torch.randn(E, H, device=DEV).bfloat16()
    wg[E // 2] = wg[0]      # a tie: the lower expert first
    x1 = torch.randn(T, H, device=DEV)
    x1[-1, 0] = float("nan") if T > 1 else 0.0      # nothing to choose in that row
    x2, l1, l2 = x1.clone(), torch.empty(T, H, device=DEV, dtype=torch.bfloat16), torch.empty(T, H, device=DEV, dtype=torch.bfloat16)
    i1, p1 = ops.resadd_moe_router(y, w, 1e-6, x1, l1, wg, k, shared, 0.75, bias)
    seqmix.norm_resadd(y, w, 1e-6, x2, l2, bias=bias)
    i2, p2 = ops.moe_router(l2, wg, k, shared, 0.75)
    assert torch.equal(x1.view(torch.int32), x2.view(torch.int32)) and torch.equal(l1.view(torch.int16), l2.view(torch.int16))
    assert torch.equal(i1, i2) and torch.equal(p1.view(torch.int32)[:-1], p2.view(torch.int32)[:-1])
    assert torch.equal(p1.isnan(), p2.isnan()) and torch.equal(p1.nan_to_num(), p2.nan_to_num())
