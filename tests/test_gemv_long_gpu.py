"""One-row GEMV with whole rows in flight (2048 < K <= 6144, one or two rows a wave) behind every epilogue: the paired ones, any number
of workgroups, K that is no whole 512s, the shortest and longest rows it takes and their neighbours outside."""
import pytest
import torch

import test_tgemm_gpu as cases
from distributed_llm_amd import ops

pytestmark = pytest.mark.gpu
KS = [2048, 2056, 2560, 4096, 4104, 6144, 6152]


@pytest.mark.parametrize("R", [1, 2])
@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("d,nq,nkv", [(64, 8, 2), (96, 3, 1), (64, 32, 4)])
def test_qkv(R, K, d, nq, nkv):
    cases.test_gemv_qkv(1, R, d, nq, nkv, K, None)


@pytest.mark.parametrize("R", [1, 2])
@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("I", [320, 2816])
def test_swiglu(R, K, I):
    cases.test_gemv_swiglu(1, R, K, I, None)


@pytest.mark.parametrize("R", [1, 2, 4])
@pytest.mark.parametrize("N,K", [(4096, 4096), (8192, 2056), (2052, 6144), (3, 2560)])
def test_plain(R, N, K):
    """A lane sums its part of K in order, however many loads travel together: the rows of a call are those of its parts."""
    torch.manual_seed(N + K)
    x, w = torch.randn(1, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    y, z = torch.empty(1, N, device="cuda").bfloat16(), torch.empty(1, N, device="cuda").bfloat16()
    ops._native(x).gemv(x, w, y, R, False)
    ops._native(x).gemv(x, w, z, 4, False)
    assert torch.equal(y, z)
    want = x.double() @ w.double().t()
    assert float((y.double() - want).norm() / want.norm()) < 2 ** -8
