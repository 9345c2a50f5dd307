"""Plans of shapes that nothing timed (ops.gemm._heuristic): runnable at every row count, and right on the GPU."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import gemm as G

SHAPES = [(1024, 1024), (1024, 2816), (5632, 1024), (4096, 1024), (4160, 64), (64, 4096), (2048, 8192), (1536, 768), (64, 64)]


@pytest.mark.parametrize("N,K", SHAPES)
def test_plans_fit_their_kernels(N, K):
    for M in range(1, 130):
        p = G._heuristic(M, N, K)
        if p[0] == "gemv":
            assert M in G._GEMV_MS and K % 8 == 0 and M * K * 2 <= 64 * 1024 and p[1] in G._GEMV_RS
        elif p[0] == "skinny":
            ntw, splits = p[1:]
            floats, tiles = G._need(M, N, K, ntw, splits)
            assert M <= G.SKINNY_MAX_M and ntw in G._NTWS and splits >= 1
            assert floats <= G.WS_FLOATS and tiles <= G.WS_COUNTERS
        else:
            assert p == ("blas",) and M > G.SKINNY_MAX_M


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", SHAPES)
def test_results(N, K):
    """f32 sums of bf16 products rounded once: within 2^-9 of the 64-bit product, and within 2^-8 with the sum's own error."""
    torch.manual_seed(N + K)
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    for M in (1, 2, 3, 4, 5, 8, 16, 17, 32, 33, 64, 65, 128):
        x = torch.randn(M, K + 8, device="cuda").bfloat16()[:, :K]
        y = G._run_plan(G._heuristic(M, N, K), x, w, False, None)
        want = x.double() @ w.double().t()
        assert float((y.double() - want).norm() / want.norm()) < 2 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(1024, 2056), (1024, 4096), (2048, 5632), (2048, 6144), (100, 6152), (2052, 5632), (1028, 4096), (7, 2816)])
@pytest.mark.parametrize("R", [1, 2, 4])
def test_gemv_long_rows(N, K, R):
    """One row on both sides of the line for whole rows in flight: 256 workgroups, 2048 < K <= 6144, the last load partly past K."""
    torch.manual_seed(N + K)
    x, w = torch.randn(1, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    y = torch.empty(1, N, device="cuda").bfloat16()
    ops._native(x).gemv(x, w, y, R, False)
    want = x.double() @ w.double().t()
    assert float((y.double() - want).norm() / want.norm()) < 2 ** -8       # one rounding to bf16, f32 sums far below


def test_rows_between_batch_sizes_take_the_next_ones_plan(monkeypatch):
    from distributed_llm_amd.engine.llm_engine import decode_buckets
    ladder = decode_buckets(1024)
    assert all(G.next_batch_size(m) == next(b for b in ladder if b >= m) for m in range(1, 1025))
    timed = {(64, 256, 512): (64, 64, 3, 4, 2, 4), (96, 256, 512): (64, 128, 3, 2, 1, 4)}
    monkeypatch.setattr(G._P, "tg_plans", timed)
    assert G.tg_plan(57, 256, 512) == G.tg_plan(64, 256, 512) == (64, 64, 3, 4, 2, 4)
    assert G.tg_plan(65, 256, 512) == (64, 128, 3, 2, 1, 4)
    assert G.tg_plan(97, 256, 512)[:3] == G.tg_plan(48, 256, 512)[:3] == (64, 64, 3)      # no plan at 128 or 48 rows: the untimed rule
    assert G.tg_slots(57, 256, 512) == 4 and G.tg_slots(70, 256, 512) == 2
