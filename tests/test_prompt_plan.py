"""Which tile a prompt's plain product takes (ops.gemm.prompt_plan): from times alone, on both sides of its line, and the products it makes."""
import pytest
import torch

from distributed_llm_amd.ops import gemm as G
from distributed_llm_amd.ops import seqmix

WIDE, SMALL = G._PP_PLANS[0], G._PP_PLANS[-1]


@pytest.fixture(autouse=True)
def none_timed(monkeypatch):
    monkeypatch.setattr(G, "_P", G._Planner())


def test_nothing_timed():
    assert G.prompt_plan(4000, 1024, 1024) is None


def timed(vendor, own):
    return [(m, t) for m, t in vendor], [(m, [t] + [1e9] * (len(G._PP_PLANS) - 1)) for m, t in own]


def test_the_faster_one_between_two_sizes():
    # 2048 columns: 64 tiles of 256 rows x 256 at 2048 rows, 128 at 4096; all of them one part-filled round
    G._P.pp_times[(2048, 1024, 0)] = timed([(1280, 90.0), (2048, 100.0), (2304, 70.0), (4096, 200.0)], [(2048, 80.0), (4096, 90.0)])
    assert G.prompt_plan(2048, 2048, 1024) == WIDE and G.prompt_plan(4096, 2048, 1024) == WIDE
    assert G.prompt_plan(2048, 2048, 1024, True) is None      # (timed without a GELU)
    assert G.prompt_plan(1100, 2048, 1024) == WIDE            # fewer rows than any timed: the vendor's time of the fewest
    assert G.prompt_plan(2049, 2048, 1024) is None and G.prompt_plan(2305, 2048, 1024) == WIDE
    assert G.prompt_plan(5120, 2048, 1024) == WIDE and G.prompt_plan(5121, 2048, 1024) is None
    G._P.pp_plans.clear()
    G._P.pp_times[(2048, 1024, 0)] = timed([(2048, 100.0), (4096, 200.0)], [(2048, 96.0), (4096, 195.0)])
    assert G.prompt_plan(2048, 2048, 1024) is None and G.prompt_plan(4096, 2048, 1024) is None
    for none in (([], []), ([(2048, 100.0)], []), ([(2048, 100.0)], [(2048, [0.0] * len(G._PP_PLANS))])):
        G._P.pp_plans.clear()
        G._P.pp_times[(2048, 1024, 0)] = none
        assert G.prompt_plan(2048, 2048, 1024) is None


def test_answers_are_bounded_and_kept_in_plan_files(tmp_path):
    G._P.pp_times[(2048, 1024, 1)] = timed([(2048, 100.0)], [(2048, 50.0)])
    for m in range(1025, 1025 + 1500):
        G.prompt_plan(m, 2048, 1024, True)
    assert len(G._P.pp_plans) <= 4097
    G._save_plans(str(tmp_path / "p.json"))
    want = dict(G._P.pp_times)
    G._P.pp_times.clear()
    G._load_plans(str(tmp_path / "p.json"))
    assert G._P.pp_times == want


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1025, 64, 64), (1300, 1600, 192), (2049, 3136, 1024), (4000, 264, 128)])
@pytest.mark.parametrize("plan", G._PP_PLANS)
def test_products(M, N, K, plan):
    torch.manual_seed(M)
    x, w = torch.randn(M, K + 8, device="cuda").bfloat16()[:, :K], (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    us = [1.0 if p == plan else 1e9 for p in G._PP_PLANS]
    for g in (0, 1):
        G._P.pp_times[(N, K, g)] = [(M, 100.0)], [(M, us)]
    want = x.double() @ w.double().t()
    got = G.linear(x, w, prompt=True)
    # f32 sums of K products, one rounding to 8 bits
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -22 * (x.abs().double() @ w.abs().double().t())).all()
    assert torch.equal(G.prompt_gelu(x, w), seqmix.gelu_erf(got))
    assert G.prompt_gelu(x[:1024], w) is None and G.prompt_gelu(x.float(), w.float()) is None


@pytest.mark.gpu
def test_timed_shapes():
    G.autotune_prompts([(256, 128, False), (256, 128, True)], "cuda")
    assert set(G._P.pp_times) == {(256, 128, 0), (256, 128, 1)}
    for vendor, own in G._P.pp_times.values():
        assert [m for m, _ in vendor] == list(G.PP_MS) and [m for m, _ in own] == list(G.PP_OWN_MS)
        assert all(t > 0 for _, t in vendor) and all(len(t) == len(G._PP_PLANS) and min(t) > 0 for _, t in own)
