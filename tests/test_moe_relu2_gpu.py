"""Squared-ReLU experts on the LDS-tiled grouped GEMM, with a shared expert among them, against a 64-bit reference.
Activations and results are each rounded once to bf16, with a relative error of at most 2^-9 an element: signs at
random, the sum over a row's activations keeps that relative size in the 2-norm, so the two together stay below 2^-8."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True, scope="module")
def _native():
    assert ops.native_available(), "HIP extension must be built for GPU tests"


# pair counts (T x 3) on both sides of the plans' lines at 128 and 1024, tiles of 64 / 128 / 256 rows full and not
@pytest.mark.parametrize("T", [1, 42, 43, 65, 341, 342, 700])
@pytest.mark.parametrize("E,H,I", [(8, 192, 128), (3, 64, 320), (63, 128, 64)])
def test_with_shared_expert(T, E, H, I):
    torch.manual_seed(T)
    x = torch.randn(T, H + 8, device=DEV).bfloat16()[:, :H]         # rows of a wider tensor
    wg = torch.randn(E, H, device=DEV).bfloat16()
    w1, w2 = (torch.randn(E + 1, a, b, device=DEV).div(b ** 0.5).bfloat16() for a, b in ((I, H), (H, I)))
    i0, p0 = ops.moe_router(x, wg, 2)
    ids, p = ops.moe_router(x, wg, 2, shared=True, scale=0.7)
    assert torch.equal(ids[:, :2], i0) and torch.equal(p[:, :2], p0 * 0.7)
    assert bool((ids[:, 2] == E).all()) and bool((p[:, 2] == 1).all())
    assert seqmix.moe_ffn_relu2_tg_ok(x, w1)
    got = seqmix.moe_ffn_relu2(x, ids, p, w1, w2)
    want = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for e in range(E + 1):
        y = torch.relu(x.double() @ w1[e].double().t()) ** 2 @ w2[e].double().t()
        want += y * (p.double() * (ids == e)).sum(1, keepdim=True)
    assert float((got.double() - want).norm() / want.norm()) < 2 ** -8


def test_router_many_experts():
    """Expert counts that are no multiple of the rows in flight, against f32 logits."""
    torch.manual_seed(3)
    for E, H in ((5, 64), (8, 1024), (61, 2048), (7, 4096), (3, 8192)):
        x, wg = torch.randn(9, H, device=DEV).bfloat16(), torch.randn(E, H, device=DEV).bfloat16()
        ids, w = ops.moe_router(x, wg, 2)
        val, idx = (x.double() @ wg.double().t()).topk(2, -1)
        assert torch.equal(ids.long(), idx)
        torch.testing.assert_close(w.double(), torch.softmax(val, -1), atol=1e-4, rtol=1e-4)
