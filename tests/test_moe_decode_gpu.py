"""Experts of few routed pairs on fragment-major weights (csrc/kernels/moe_decode.hip): the bits of the grouped GEMM, at edges of the
row groups and of the pair list, for every end of the layer."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix

DEV = "cuda"


def _case(T, E, k, H, I, mode, same):
    torch.manual_seed(T + E + H)
    x = torch.randn(T, H, device=DEV).bfloat16()
    ids = torch.stack([torch.randperm(E + 1, device=DEV)[:k] for _ in range(T)]).to(torch.int32)      # (E: an identity expert, clamped)
    if same:
        ids[:, 0] = E - 1      # one expert runs every row
    wts = torch.rand(T, k, device=DEV)
    w1 = (torch.randn(E, I if mode else 2 * I, H, device=DEV) * H ** -0.5).bfloat16()
    w2 = (torch.randn(E, H, I, device=DEV) * I ** -0.5).bfloat16()
    frag = (ops.frag_experts(w1, paired=not mode), ops.frag_experts(w2))
    run = (lambda **kw: seqmix.moe_ffn_relu2(x, ids, wts, w1, w2, **kw)) if mode else (lambda **kw: ops.moe_ffn_tg(x, ids, wts, w1, w2, **kw))
    return x, ids, wts, w1, w2, frag, run


@pytest.fixture(autouse=True)
def all_sizes(monkeypatch):
    monkeypatch.setattr(ops, "MOE_FEW_TOKENS", 256)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("T,E,k,H,I", [(1, 8, 2, 1024, 1024), (5, 3, 2, 64, 192), (12, 8, 2, 1024, 1024), (17, 4, 3, 320, 64), (33, 9, 3, 1024, 512),
                                       (64, 8, 2, 128, 256), (64, 64, 4, 192, 128), (85, 2, 3, 64, 64)])
@pytest.mark.parametrize("same", [False, True])
def test_bits_of_the_grouped_gemm(mode, T, E, k, H, I, same):
    x, ids, wts, w1, w2, frag, run = _case(T, E, k, H, I, mode, same)
    plan = {} if mode else dict(plan=ops.MOE_PLANS["decode"])
    want, got, four = run(**plan), run(frag=frag + (True,)), run(frag=frag)
    assert ops.moe_few(x, ids, frag) and torch.isfinite(got.float()).all()
    # K in four parts: other f32 sums, so bf16 roundings of the activations and the outputs
    assert (four.float() - want.float()).norm() <= 2.0 ** -8 * want.float().norm()
    if mode and T * k > 128:      # (another plan's product: no chain of its own)
        torch.testing.assert_close(got.float(), want.float(), atol=2e-2, rtol=2e-2)
    else:
        assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("T", [3, 24])
@pytest.mark.parametrize("steps", range(1, 14))
def test_stages_of_a_quarter(mode, T, steps):
    """A wave's quarter of K ends in a first, second or third stage, whole and not, and the last waves have less of it or none."""
    for K in (128 * steps, 128 * steps - 64):
        test_bits_of_the_grouped_gemm(mode, T, 2, 2, K, K, True)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("T,groups", [(1, 1), (24, 4), (40, 1)])
def test_sum_ends_in_the_stream(mode, T, groups):
    x, ids, wts, w1, w2, frag, run = _case(T, 9, 3, 1024, 256, mode, False)
    w, s = torch.rand(1024, device=DEV) + 0.5, torch.randn(T, 1024, device=DEV)
    out = []
    for kw in ({}, dict(frag=frag + (True,))):
        xs, xl = s.clone(), torch.empty(T, 1024, dtype=torch.bfloat16, device=DEV)
        assert run(tail=(w, 1e-6, xs, xl, groups), **kw) is None
        out.append((xs, xl))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 12, 64])
def test_sum_added_to_the_residual(T):
    x, ids, wts, w1, w2, frag, _ = _case(T, 8, 2, 1024, 256, 0, False)
    r0, out = torch.randn(T, 1024, device=DEV).bfloat16(), []
    for f in (None, frag + (True,)):
        r, ssq = r0.clone(), torch.zeros(2, T, device=DEV)
        n = ops.moe_ffn_tg_resadd(x, ids, wts, w1, w2, r, ssq, frag=f)
        out.append((r, ssq[:n]))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


class _Fragments:
    """frag_experts' shape of weights, without the weights."""
    def __init__(self, E, N, K):
        self.shape, self.numel = (E, N // 16, K // 32, 64, 8), lambda: E * N * K


@pytest.mark.parametrize("E,k,H,I,order,tokens", [(8, 2, 1024, 1024, False, 64), (8, 2, 1024, 1024, True, 64), (8, 2, 4096, 3584, False, 40), (8, 2, 4096, 3584, True, 40),
                                                  (2, 2, 1024, 1024, False, 64), (2, 2, 1024, 1024, True, 24), (64, 4, 2048, 1408, False, 64),
                                                  (4, 2, 4096, 3584, False, 20), (1, 1, 512, 512, True, 24), (8, 8, 256, 256, False, 32)])
def test_how_many_are_few(monkeypatch, E, k, H, I, order, tokens):
    """The most tokens that run on the fragment-major copies: of large experts, and of one wave a tile, by the pairs an expert has."""
    monkeypatch.setattr(ops, "MOE_FEW_TOKENS", 64)
    frag = (_Fragments(E, 2 * I, H), _Fragments(E, H, I)) + ((True,) if order else ())
    few = lambda T: ops.moe_few(torch.zeros(T, 8, dtype=torch.bfloat16), torch.zeros(T, k, dtype=torch.int32), frag)  # noqa: E731
    assert few(1)["few_ks"] == few(tokens)["few_ks"] == (1 if order else 4) and few(tokens + 1) == {} and few(0) == {}
