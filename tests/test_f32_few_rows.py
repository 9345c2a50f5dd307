"""f32 products of at most eight rows (csrc/kernels/f32_gemm.hip) against a double's: rows that fill no block of four, both sides of the lines between
waves and steps in flight, waves without a step, columns past N, rows of a wider matrix, rows that are not finite."""
import pytest
import torch

from distributed_llm_amd.ops import gemm as G


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("N,K", [(16, 16), (50, 80), (500, 512), (515, 528), (1000, 1040), (96, 4096), (4080, 4096), (4100, 4112), (33, 8192)])
def test_against_64_bits(M, N, K):
    torch.manual_seed(M + N + K)
    x, w = torch.randn(M, K + 4, device="cuda")[:, :K], torch.randn(N, K, device="cuda")
    wf = G.frag_weight(w)
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    # a sum's roundings: at most K / 32 + 4 terms one behind the other, two for the groups, sixteen for the waves (nine rows: K / 8 + 24)
    bound = (K / (32 if M <= 8 else 8) + 24) * 2.0 ** -24 * size
    got = G.f32_linear(x, wf, N)
    assert ((got.double() - want).abs() <= bound).all()
    # (slope at most 1.13; four roundings of a value or of 1)
    assert ((G.f32_linear(x, wf, N, gelu=True).double() - torch.nn.functional.gelu(want)).abs() <= 1.13 * bound + 4 * 2.0 ** -24 * (want.abs() + 1)).all()
    if M > 1:
        x[M - 1, K - 1] = float("nan")
        bad = G.f32_linear(x, wf, N)
        assert torch.equal(bad[:-1], got[:-1]) and bad[-1].isnan().all()


def test_rows_it_is_for():
    rows = lambda M, K: torch.zeros(M, K)  # noqa: E731
    assert all(G.fg_takes(rows(M, 4096), N) for M in (1, 8) for N in (64, 32000))
    assert not any(G.fg_takes(rows(M, 4096), 1024) for M in (9, 16)) and G.fg_takes(rows(16, 2048), 1024)
