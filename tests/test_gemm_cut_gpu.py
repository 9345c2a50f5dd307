"""Untimed products whose splits of K stay in workgroups of their own, or share one: the same bits, whatever the rows and the columns
of a workgroup."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import gemm

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True, scope="module")
def _native():
    assert ops.native_available(), "HIP extension must be built for GPU tests"


@pytest.mark.parametrize("N,K", [(128, 2048), (64, 4096), (144, 8192), (256, 8192), (512, 2048), (528, 2048), (3000, 1536), (3000, 4096), (2800, 8192)])
def test_same_bits(N, K):
    torch.manual_seed(N)
    w, x = (torch.randn(m, K, device="cuda").bfloat16() for m in (N, 64))
    splits = gemm._heuristic(64, N, K)[2]
    want = gemm._run_plan(("skinny", 2, splits), x, w, False, None)
    assert float((want.double() - x.double() @ w.double().t()).norm() / want.double().norm()) < 2 ** -8
    for M in (1, 2, 3, 16, 17, 32, 33, 64):
        assert torch.equal(gemm.linear(x[:M], w), want[:M])
