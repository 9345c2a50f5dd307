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


def test_sizes_that_an_engine_has_no_rows_for_are_not_timed():
    left = lambda most, have=(): G._pp_left((1280, 2048, 4096, 8192), [(m, 1.0) for m in have], most)  # noqa: E731
    assert left(1025) == left(1280) == [1280] and left(1281) == left(2048) == [1280, 2048] and left(9000) == [1280, 2048, 4096, 8192]
    assert left(2000, (1280, 2048)) == [] and left(2049, (1280, 2048)) == [4096]      # what was timed stands


class Timing:
    """Stands in for the device and its clock; memory for tensors of ``rows``."""

    def __init__(self, monkeypatch, rows=1 << 20):
        self.rows, self.seen = rows, []
        randn = torch.randn

        def made(*s, dtype=None, device=None):
            if s[0] > self.rows:
                raise torch.OutOfMemoryError("no room")
            self.seen.append(s[0])
            return randn(1, 1)
        monkeypatch.setattr(torch, "randn", made)
        monkeypatch.setattr(torch, "empty", lambda *s, **k: None)
        monkeypatch.setattr(G, "_sk_grid", lambda d: 256)
        monkeypatch.setattr(G, "_native", lambda t: None)
        monkeypatch.setattr(G, "_time", lambda f, iters: 100.0)


def test_an_engine_times_what_it_can_hold(monkeypatch):
    t = Timing(monkeypatch)
    G.autotune_prompts([(1024, 512, False)], "cuda", 1024)
    assert not t.seen and not G._P.pp_times
    G.autotune_prompts([(1024, 512, False)], "cuda", 1500)
    assert [m for m, _ in G._P.pp_times[(1024, 512, 0)][0]] == [1280, 1536] and [m for m, _ in G._P.pp_times[(1024, 512, 0)][1]] == [2048]
    assert G.prompt_plan(1500, 1024, 512) is None and G.prompt_plan(9000, 1024, 512) is None
    first, G._P.pp_times[(1024, 512, 0)][0][0] = G._P.pp_times[(1024, 512, 0)], (1280, 77.0)
    t.seen.clear()
    G.autotune_prompts([(1024, 512, False)], "cuda", 1 << 20)      # a larger engine times the rest
    vendor, own = G._P.pp_times[(1024, 512, 0)]
    assert vendor is first[0] and vendor[0] == (1280, 77.0) and [m for m, _ in vendor] == list(G.PP_MS) and [m for m, _ in own] == list(G.PP_OWN_MS)
    assert t.seen.count(1280) == t.seen.count(2048) - 1 == 0 and (9000, 1024, 512, 0) not in G._P.pp_plans


@pytest.mark.parametrize("rows,vendor,own", [(5000, 4864, 4096), (1500, 1280, None), (600, None, None)])
def test_sizes_without_memory_are_left_to_the_vendor(monkeypatch, rows, vendor, own):
    Timing(monkeypatch, rows)
    G.autotune_prompts([(1024, 512, False), (256, 128, True)], "cuda")
    for key in ((1024, 512, 0), (256, 128, 1)):
        a, b = G._P.pp_times[key]
        if key[0] > rows:      # no room for its weights either
            assert not a and not b
            continue
        assert (a[-1][0] if a else None) == (vendor if vendor else None) and (b[-1][0] if b else None) == own
    assert G.prompt_plan(12000, 1024, 512) is None


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
