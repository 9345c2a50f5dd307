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


def test_untimed_tiles(monkeypatch):
    """Both sides of each line of the rule for shapes that nobody timed."""
    _none_timed(monkeypatch)
    monkeypatch.setattr(G._P, "cus", 256)
    tile = lambda M, N, K: G.tg_plan(M, N, K)[:2]  # noqa: E731
    assert tile(3200, 384, 1536) == (64, 128) and tile(3136, 384, 1536) == (64, 64)      # 150 and 147 tiles
    assert tile(600, 2304, 768) == (64, 64) and tile(640, 2432, 768) == (64, 128)         # 180 and 190, more columns than rows
    assert tile(4000, 1024, 4096) == (128, 128) and tile(2000, 1024, 4096) == tile(4200, 1024, 4096) == (64, 128)
    assert tile(16000, 768, 3072) == (128, 128) and tile(8000, 768, 3072) == (64, 128)
    assert tile(4000, 1024, 1984) == tile(16000, 4096, 1024) == tile(1000, 8192, 2048) == (64, 128)
    monkeypatch.setattr(G._P, "cus", 128)
    assert tile(2000, 1024, 4096) == (128, 128)


def test_expert_tiles(monkeypatch):
    """Both sides of each line of the rule for an expert layer's tiles: pairs, pairs an expert, CUs that each product's tiles fill."""
    from distributed_llm_amd import ops
    monkeypatch.setattr(G._P, "cus", 256)

    def plan(pairs, E, N1, N2):
        w1, w2 = torch.empty(E, N1, 64, device="meta"), torch.empty(E, N2, N1 // 2, device="meta")
        return next(k for k, v in ops.MOE_PLANS.items() if v == ops.moe_plan(pairs, w1, w2))

    assert [plan(p, 8, 14336, 4096) for p in (128, 129, 1024, 1025)] == ["decode", "mid", "mid", "wide"]
    assert ops.moe_plan(5000) == ops.MOE_PLANS["prefill"]      # (no weights: by the pairs alone)
    assert [plan(p, 64, 2048, 2048) for p in (64 * 128 - 1, 64 * 128)] == ["mid", "wide"]
    # 8 experts of 1024 x 1024: 17.6 row tiles of the first product's 8 columns are 0.55 of the CUs, 32 of the second's 4 are half
    assert [plan(p, 8, 2048, 1024) for p in (3481, 3482, 7167, 7168)] == ["mid", "prefill", "prefill", "wide"]
    monkeypatch.setattr(G._P, "cus", 128)
    assert [plan(p, 8, 2048, 1024) for p in (3000, 3482)] == ["prefill", "wide"]


def _timed(monkeypatch, N, K, us, small):
    """Tables as the autotuner leaves them: a round of 256 tiles of 256 x 256 and of 256 x 128, and plans of small tiles."""
    big, half = (256, 256, 2, 1, 1, 8), (256, 128, 3, 1, 1, 8)
    times = [(p, m, u * -(-(-(-m // 256) * -(-N // p[1])) // 256)) for p, u in ((big, us), (half, 0.6 * us)) for m in (2048, 4096, 8192)]
    monkeypatch.setattr(G._P, "pf_times", {(N, K): times})
    monkeypatch.setattr(G._P, "pf_small", {(m, N, K): ((128, 128, 3, 1, 1, 8), small) for m in G.PF_SMALL_MS})
    monkeypatch.setattr(G._P, "pf_parts", {})
    monkeypatch.setattr(G._P, "tg_plans", {(m, N, K): big for m in (2048, 4096, 8192)})
    return big, half


@pytest.mark.parametrize("N,us,small", [(2048, 90.0, 15.0), (2560, 90.0, 15.0), (11264, 70.0, 20.0), (96, 50.0, 10.0), (2048, 20.0, 60.0)])
def test_prompt_parts(monkeypatch, N, us, small):
    big, half = _timed(monkeypatch, N, 256, us, small)
    for M in list(range(1025, 12000, 331)) + [8192, 8928, 9000, 40000]:
        parts = G.prompt_parts(M, N, 256)
        assert sum(r for r, _ in parts) == M and len(parts) <= 2 and all(r > 0 for r, _ in parts)
        (rows, plan) = parts[0]
        assert plan in (big, half)
        if len(parts) == 2:      # whole rounds of large tiles, then rows the small plans were timed for
            assert rows % plan[0] == 0 and parts[1][0] <= G.PF_SMALL_MS[-1]
            tiles, every = rows // plan[0] * -(-N // plan[1]), -(-M // plan[0]) * -(-N // plan[1])
            assert -(-tiles // 256) < -(-every // 256)
    if (N, us) == (2048, 90.0):
        assert G.prompt_parts(8928, N, 256) == ((8192, big), (736, (128, 128, 3, 1, 1, 8)))
        assert G.prompt_parts(8192, N, 256) == ((8192, big),)
    monkeypatch.setattr(G._P, "pf_times", {})
    monkeypatch.setattr(G._P, "pf_parts", {})
    assert G.prompt_parts(8928, N, 256) is None


def test_vendor_core_by_the_rows_at_hand(monkeypatch):
    """Times as TinyLlama's down product has them: one round of 256 x 256 tiles at 8192 rows beats the vendor's product, two at 10000 do not,
    two full ones do again; a bucket's own choice stands, and rows that nothing was timed for go by their bucket."""
    monkeypatch.delenv("DLLM_FUSED_CORE", raising=False)
    _none_timed(monkeypatch)
    N, K, wide = 2048, 5632, (256, 256, 2, 1, 1, 4)
    monkeypatch.setattr(G._P, "cus", 256)
    G._P.pf_times[N, K] = [(wide, m, t) for m, t in ((2048, 120.0), (4096, 122.0), (8192, 137.0))]
    G._P.pf_lin[N, K] = [(1280, 45.0), (2048, 53.0), (4096, 86.0), (6144, 118.0), (8192, 140.0), (10240, 205.0), (12288, 250.0), (16384, 298.0)]
    G._P.tg_plans.update({(m, N, K): wide for m in G.PREFILL_MS})
    G._P.pf_small.update({(m, N, K): ((128, 128, 3, 1, 1, 8), 30.0) for m in G.PF_SMALL_MS})
    G._P.fused_core.update({(2048, N, K): "lin", (4096, N, K): "lin", (8192, N, K): "tg"})
    want = {1100: True, 2048: True, 4096: True, 4500: True, 6000: True, 8000: False, 8192: False, 8900: False, 10000: True, 11679: True,
            12288: True, 13000: False, 16384: False, 20000: True}
    for _ in range(2):      # (worked out, then looked up)
        assert {M: G.use_vendor_core(M, N, K) for M in want} == want
    parts = lambda M: [p == "lin" for _, _, p in G._row_parts(M, N, K)]  # noqa: E731
    assert parts(10000) == [True] and parts(8900) == [False, False] and parts(16000) == [False]
    # a choice is kept unless the other form is shorter by more than the times are uncertain by
    G._P.fused_core[8192, N, K] = "lin"
    G._P.pf_vendor.clear()
    assert G.use_vendor_core(8000, N, K) and G.use_vendor_core(10000, N, K) and not G.use_vendor_core(8900, N, K)
    G._P.fused_core[8192, N, K] = "tg"
    for gone in ("pf_lin", "pf_times"):
        monkeypatch.setattr(G._P, gone, {})
        monkeypatch.setattr(G._P, "pf_vendor", {})
        assert not G.use_vendor_core(10000, N, K) and G.use_vendor_core(3000, N, K)


def test_rows_that_do_not_fit_are_not_timed(monkeypatch):
    """Beside a large model and its pool the largest row counts may find no memory: they are left out, and the engine starts."""
    _none_timed(monkeypatch)
    monkeypatch.setattr(G, "PREFILL_MS", (2048,))
    monkeypatch.setattr(G, "PF_SMALL_MS", ())
    monkeypatch.setattr(G, "PF_LIN_MS", (1280, 12288, 16384))

    def call(role, x, *a):
        if x.shape[0] > 12000:
            raise torch.OutOfMemoryError("no memory")
        return lambda i: None
    monkeypatch.setattr(G, "_fused_call", call)
    monkeypatch.setattr(G, "_native", lambda x: None)
    monkeypatch.setattr(G, "_time", lambda fn, iters=24: 7.0)
    G._autotune_prefill([(64, 64)], "cpu", False, {(64, 64): "resadd"})
    assert G._P.pf_lin == {(64, 64): [(1280, 7.0), (2048, 7.0)]} and set(G._P.fused_core) == {(2048, 64, 64)}


@pytest.mark.gpu
@pytest.mark.parametrize("panel", [False, True])
def test_parts_are_the_whole(monkeypatch, panel):
    """Each fused product in two parts against one launch: every row's chain over K is the same, so are its bits."""
    torch.manual_seed(1)
    M, H, I, nq, nkv, d = 1300, 256, 512, 4, 2, 64
    N = (nq + 2 * nkv) * d
    rnd = lambda *s: (torch.randn(*s, device="cuda") * s[-1] ** -0.5).bfloat16()  # noqa: E731
    r, w_qkv, w_gu, w_d, res = rnd(M, H), rnd(N, H), rnd(2 * I, H), rnd(H, I), rnd(M, H)
    ssq = torch.rand(1, M, device="cuda") + 1.0      # (several partial sums are added in an order that depends on the tile)
    pos = torch.randint(0, 2000, (M,), device="cuda", dtype=torch.int32)
    slots = torch.randperm(1600, device="cuda")[:M].to(torch.int32)
    cs = ops.rope_cos_sin(2048, d, 10000.0, "cuda")
    wp = G.panel_weight if panel else (lambda w: None)

    def run():
        kc, vc = torch.zeros(100, nkv, 16, d, device="cuda").bfloat16(), torch.zeros(100, nkv, d, 16, device="cuda").bfloat16()
        q = G.qkv_rope_cache(r, w_qkv, ssq, 1, 1e-5, pos, cs, slots, kc, vc, nq, nkv, d, wp=wp(w_qkv))
        act = G.swiglu_matmul(r, w_gu, ssq, 1, 1e-5, wp=wp(w_gu))
        x, so = res.clone(), torch.full((G.max_slots(H, M), M), float("nan"), device="cuda")
        n = G.matmul_resadd(act, w_d, x, so, wp=wp(w_d))
        return q, kc, vc, act, x, so[:n].sum(0)

    big, small = (256, 256, 2, 1, 1, 8), (64, 128, 3, 1, 1, 8)
    monkeypatch.setattr(G, "use_vendor_core", lambda M, N, K: False)
    monkeypatch.setattr(G, "prompt_parts", lambda M, N, K: ((M, big),))
    one = run()
    monkeypatch.setattr(G, "prompt_parts", lambda M, N, K: ((1024, big), (M - 1024, small)))
    two = run()
    assert all(torch.equal(a, b) for a, b in zip(one[:5], two[:5]))
    torch.testing.assert_close(one[5], two[5], rtol=1e-5, atol=1e-6)
    monkeypatch.setattr(G, "use_vendor_core", lambda M, N, K: True)
    for a, b in zip(one, run()):
        torch.testing.assert_close(a.float(), b.float(), rtol=2e-2, atol=2e-2)


def test_decode_gemm_in_place_of_a_skinny_plan(monkeypatch):
    """A timed plan runs as timed, unless the decode GEMM was faster, has to keep the order of its sums or saves the activation's launch; and
    only where its slabs, one column of a tile wider than the skinny plan's, fit the workspace."""
    monkeypatch.setattr(G._P, "plans", {(16, 2048, 2048, False): ("skinny", 2, 8), (64, 32000, 2048, False): ("skinny", 2, 8),
                                        (8, 2048, 2048, False): ("tg", 64, 64, 3, 1, 1, 4), (4, 2048, 2048, False): ("skinny", 4, 2)})
    monkeypatch.setattr(G._P, "dg_plans", {(8, 2048, 2048): (1, 2, 4)})
    of = lambda M, N, K, *a, **k: G._linear_plan(torch.empty(M, K), torch.empty(N, K), *a, **k)  # noqa: E731
    assert of(16, 2048, 2048, True, False) == (("skinny", 2, 8), 1, None)
    assert of(16, 2048, 2048, True, True)[2] == of(16, 2048, 2048, True, False, ends=True)[2] == (2, 2, 8)
    assert of(4, 2048, 2048, True, True)[2] == (2, 2, 2) and of(4, 2048, 2048, True, False)[2] is None
    assert of(8, 2048, 2048, True, False)[2] == (1, 2, 4) and of(8, 2048, 2048, True, True)[2] is None
    assert G._need(64, 32000, 2048, 2, 8)[0] <= G.WS_FLOATS < G._need_dg(64, 32000, 2048, (2, 2, 8))[0]
    for keep in (False, True):
        assert of(64, 32000, 2048, True, keep, ends=True) == (("skinny", 2, 8), 1, None)
    # nothing timed: the rule's plan, its splits together, with and without copies
    plan = G._heuristic(16, 1024, 1024)
    assert of(16, 1024, 1024, False, False) == (plan, G._splits_together(16, 1024, 1024, plan), None)
    assert of(16, 1024, 1024, True, False)[2] == (plan[1], G._splits_together(16, 1024, 1024, plan), plan[2])
    for M in range(1, 65):
        for N, K in SHAPES:
            dg = of(M, N, K, True, False)[2]
            assert dg is None or G._need_dg(M, N, K, dg)[0] <= G.WS_FLOATS


def _none_timed(monkeypatch):
    for name in ("plans", "tg_plans", "dg_plans", "fused_core", "frag_core", "fused_opts", "pf_times", "pf_small", "pf_parts", "pf_lin", "pf_vendor"):
        monkeypatch.setattr(G._P, name, {})


def test_cores_with_and_without_copies(monkeypatch):
    """One process serves models with and without fragment-major copies of the same shapes: the decode GEMM runs where there is a copy and
    the rows are as it reads them; everything else gets what was chosen without it."""
    monkeypatch.delenv("DLLM_FUSED_CORE", raising=False)
    _none_timed(monkeypatch)
    N, K = 2048, 2048
    rows = lambda M: torch.zeros(M, K + 8, dtype=torch.bfloat16)[:, :K]  # noqa: E731
    odd = torch.zeros(2, K + 4, dtype=torch.bfloat16)[:, :K]
    G._P.fused_core.update({(1, N, K): "gemv2", (2, N, K): "lin", (16, N, K): "skE4", (64, N, K): "tg", (32, N, K): "tg"})
    G._P.frag_core.update({(1, N, K): "dg1.2.2", (2, N, K): "dg1.1.4", (16, N, K): "dg2.2.2", (64, N, K): "dg1.1.2", (32, N, K): "lin"})
    wf = torch.zeros(1)
    assert [G.fused_dg(rows(M), N, K, wf) for M in (1, 2, 16, 32, 57, 64)] == [(1, 2, 2), (1, 1, 4), (2, 2, 2), None, (1, 1, 2), (1, 1, 2)]
    assert all(G.fused_dg(rows(M), N, K, None) is None for M in (1, 2, 16, 32, 57, 64))
    assert G.fused_dg(odd, N, K, wf) is None and G.use_vendor_core(2, N, K, True)
    for frag in (False, True):      # (with copies: rows that the decode GEMM does not read)
        assert G.fused_gemv_r(rows(1), N, frag) == 2 and G.fused_ske(rows(16), N, K, frag) == 4 and not G.use_vendor_core(64, N, K, frag)
    assert G.use_vendor_core(32, N, K, True) and not G.use_vendor_core(32, N, K)
    G._P.frag_core[(1, N, K)] = "skE2"      # chosen among more: not what is chosen without
    assert G.fused_ske(rows(1), N, K, True) == 2 and G.fused_gemv_r(rows(1), N, True) == 0 and G.fused_gemv_r(rows(1), N) == 2


def test_narrow_producers_and_their_consumers(monkeypatch):
    _none_timed(monkeypatch)
    shapes = [(2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632)]
    prod, cons = [(M,) + shapes[1] for M in (1, 4, 8)], [(M,) + shapes[2] for M in (1, 4, 8)]
    G._P.fused_core.update({prod[0]: "gemv2", cons[0]: "tg", prod[1]: "lin", cons[1]: "tg", prod[2]: "gemv1", cons[2]: "skE2"})
    G._P.frag_core.update({prod[0]: "gemv2", cons[0]: "dg2.1.1", prod[1]: "dg1.2.2", prod[2]: "dg1.1.4", cons[2]: "tg"})
    for k in prod:
        G._P.fused_opts[k] = {"gemv2": 3.0, "gemv1": 3.1, "dg1.2.2": 3.2, "dg1.1.4": 3.3, "dg2.1.1": 4.0, "lin": 5.0}
    G._couple_gemv_choices(shapes, [1, 4, 8], verbose=False)
    assert [G._P.fused_core[k] for k in prod] == ["lin", "lin", "gemv1"]
    assert [G._P.frag_core[k] for k in prod] == ["gemv2", "dg2.1.1", "dg2.1.1"]      # a consumer timed without copies counts, too


def test_plan_file(monkeypatch, tmp_path):
    """What was timed comes back; a file that kept one choice for weights with and without copies has its decode GEMMs timed again."""
    import json
    _none_timed(monkeypatch)
    k = (16, 2048, 2048)
    G._P.plans[k + (False,)] = ("skinny", 2, 4)
    G._P.tg_plans[k], G._P.fused_core[k], G._P.frag_core[k] = (64, 64, 3, 1, 1, 4), "skE4", "dg1.2.2"
    G._P.dg_plans.update({k: (1, 2, 4), (8, 2048, 2048): None})
    G._P.pf_times[2048, 2048], G._P.pf_small[128, 2048, 2048] = [((256, 256, 2, 1, 1, 8), 2048, 50.0)], ((64, 64, 3, 1, 1, 4), 9.0)
    G._P.pf_lin[2048, 2048] = [(2048, 40.0), (3072, 55.0)]
    tables = ("plans", "tg_plans", "dg_plans", "fused_core", "frag_core", "pf_times", "pf_small", "pf_lin")
    want = {n: dict(getattr(G._P, n)) for n in tables}
    G._save_plans(str(tmp_path / "sub" / "plans.json"))
    _none_timed(monkeypatch)
    G._load_plans(str(tmp_path / "sub" / "plans.json"))
    assert {n: getattr(G._P, n) for n in tables} == want
    _none_timed(monkeypatch)
    with open(tmp_path / "old.json", "w") as f:
        json.dump({"c,16,2048,2048": "dg1.2.2", "c,8,2048,2048": "tg", "d,8,2048,2048": [1, 2, 4]}, f)
    G._load_plans(str(tmp_path / "old.json"))
    assert G._P.fused_core == {(8, 2048, 2048): "tg"} and G._P.dg_plans == {(8, 2048, 2048): (1, 2, 4)} and not G._P.frag_core


def test_plan_file_of_other_code(monkeypatch, tmp_path):
    """Times hold for the kernels and candidates that were timed: nothing comes back from a file that was timed with others, or does not say."""
    import json
    from types import SimpleNamespace
    _none_timed(monkeypatch)
    card = lambda name, cus: SimpleNamespace(name=name, gcnArchName="gfx950", multi_processor_count=cus)
    cards = {0: card("A", 256), 1: card("A", 64), 2: card("", 256)}
    monkeypatch.setattr(torch.cuda, "get_device_properties", lambda d: cards[d])
    built = tmp_path / "kernels.so"
    monkeypatch.setattr(G, "_load_ext", lambda: SimpleNamespace(__file__=str(built)))
    made = []
    for content, card in ((b"one", 0), (b"two", 0), (b"one", 1)):
        built.write_bytes(content)
        made.append(G._timed_with(card))
    assert len(set(made)) == 3 and built.write_bytes(b"one") and G._timed_with(0) == made[0] == G._timed_with(2)      # (a profiler hides the name)
    k, path = (16, 2048, 2048), str(tmp_path / "plans.json")
    G._P.tg_plans[k] = (64, 64, 3, 1, 1, 4)
    G._save_plans(path, made[0])
    for m, want in ((made[1], {}), (made[0], {k: (64, 64, 3, 1, 1, 4)})):
        G._P.tg_plans.clear()
        G._load_plans(path, m)
        assert G._P.tg_plans == want
    with open(path) as f:
        d = json.load(f)
    with open(path, "w") as f:
        json.dump({k: v for k, v in d.items() if k.startswith("t,")}, f)
    G._P.tg_plans.clear()
    G._load_plans(path, made[0])
    assert not G._P.tg_plans


@pytest.mark.gpu
def test_old_plan_file_is_timed_again(monkeypatch, tmp_path):
    import json
    _none_timed(monkeypatch)
    monkeypatch.setattr(G, "PREFILL_TUNE", False)
    path, key = str(tmp_path / "plans.json"), "%d,%d,%d,0" % (4, 1024, 768)
    with open(path, "w") as f:
        json.dump({key: ["skinny", 1, 1], "%d,%d,%d,0" % (4, 999, 768): ["blas"]}, f)
    monkeypatch.setenv("DLLM_GEMM_PLANS", path)
    G.autotune([(1024, 768, False)], [4], "cuda")
    assert set(G._P.plans) == {(4, 1024, 768, False)}
    timed = dict(G._P.plans)
    _none_timed(monkeypatch)
    monkeypatch.setattr(G, "_time", lambda *a, **k: pytest.fail("timed again"))
    G.autotune([(1024, 768, False)], [4], "cuda")
    assert G._P.plans == timed


@pytest.mark.gpu
def test_copies_are_timed_when_they_come_second(monkeypatch):
    """Shapes timed for a model without copies, then for one with them: the decode GEMM is timed, the earlier choices stand."""
    _none_timed(monkeypatch)
    monkeypatch.delenv("DLLM_FUSED_CORE", raising=False)
    monkeypatch.delenv("DLLM_GEMM_PLANS", raising=False)
    monkeypatch.setattr(G, "PREFILL_TUNE", False)
    fused = [(1024, 1024), (1024, 768), (2816, 1024), (1024, 1408)]
    tune = lambda frag: G.autotune([(n, k, False) for n, k in fused], [4, 96], "cuda", fused=fused, qkv_dims=(12, 2, 64), frag=frag)  # noqa: E731
    tune([])
    assert not G._P.frag_core and not G._P.dg_plans and all(not c.startswith("dg") for c in G._P.fused_core.values())
    kept = dict(G._P.fused_core), dict(G._P.plans), dict(G._P.tg_plans)
    tune(fused)
    assert (G._P.fused_core, G._P.plans, G._P.tg_plans) == kept
    assert set(G._P.dg_plans) == set(G._P.frag_core) == {(4,) + f for f in fused}
    assert all(any(c.startswith("dg") for c in G._P.fused_opts[(4,) + f]) for f in fused)


@pytest.mark.parametrize("role", ["resadd", None])
def test_refused_prompt_plans(monkeypatch, role):
    """A plan that the product takes and its epilogue refuses, one that both refuse and small plans that are refused: left out, and nothing
    that timing forced for them stays behind."""
    _none_timed(monkeypatch)
    N, K = 128, 64
    monkeypatch.setattr(G, "PREFILL_MS", (2048, 4096))
    monkeypatch.setattr(G, "_native", lambda x: None)
    monkeypatch.setattr(G, "_post_us", lambda *a: 3.0)
    us = {p: 50.0 + i for i, p in enumerate(dict.fromkeys(G._PF_PLANS + G._PF_SMALL))}
    us[G._PF_PLANS[3]] = 10.0      # the fastest product: its epilogue is refused
    ran = []

    def tgemm(ext, x, w, epi, plan, **kw):
        M = x.shape[0]
        if M == 256 or (plan != G._PF_SMALL[0] if M in G.PF_SMALL_MS else plan == G._PF_PLANS[1]):
            raise RuntimeError("no such plan")
        ran.append(us[plan])

    def whole(i):
        (_, plan), = G.prompt_parts(ran_rows[-1], N, K)
        assert not G.use_vendor_core(ran_rows[-1], N, K)
        if plan == G._PF_PLANS[3]:
            raise RuntimeError("no such epilogue")
        ran.append(us[plan] + 5.0)

    ran_rows = []
    monkeypatch.setattr(G, "_fused_call", lambda role, x, *a: ran_rows.append(x.shape[0]) or (whole if role else None))
    monkeypatch.setattr(G, "_tgemm", tgemm)
    monkeypatch.setattr(G, "_time", lambda fn, iters=24: (ran.append(1e3), fn(0), ran[-1])[-1])
    G._autotune_prefill([(N, K)], torch.device("cpu"), False, {(N, K): role} if role else {})
    out = {G._PF_PLANS[1]} | ({G._PF_PLANS[3]} if role else set())
    extra = 5.0 if role else 0.0
    assert G._P.pf_times[N, K] == [(p, M, us[p] + extra) for M in (2048, 4096) for p in G._PF_PLANS if p not in out]
    assert G._P.tg_plans == {(M, N, K): G._PF_PLANS[0 if role else 3] for M in (2048, 4096)}
    assert set(G._P.fused_core) == {(2048, N, K), (4096, N, K)} and not G._P.pf_parts
    assert set(G._P.pf_small) == {(M, N, K) for M in G.PF_SMALL_MS if M != 256}


@pytest.mark.parametrize("cus", [64, 128, 256, 304])
def test_prompt_parts_by_the_devices_cus(monkeypatch, cus):
    """Rounds are over the CUs of the device at hand: two rounds and an eighth of one more become two, and a launch of small tiles."""
    N, big, small = 2048, (256, 256, 2, 1, 1, 8), (128, 128, 3, 1, 1, 8)
    monkeypatch.setattr(G._P, "cus", cus)
    rows = lambda rounds: int(rounds * cus) // 8 * 256  # noqa: E731
    monkeypatch.setattr(G._P, "pf_times", {(N, 256): [(big, rows(2), 180.0)]})
    monkeypatch.setattr(G._P, "pf_small", {(m, N, 256): (small, 10.0) for m in G.PF_SMALL_MS})
    monkeypatch.setattr(G._P, "tg_plans", {(m, N, 256): big for m in G.PREFILL_MS})
    monkeypatch.setattr(G._P, "pf_parts", {})
    tail = rows(2.125) - rows(2)
    assert G.prompt_parts(rows(2), N, 256) == ((rows(2), big),)
    assert tail > G.PF_SMALL_MS[-1] or G.prompt_parts(rows(2) + tail, N, 256) == ((rows(2), big), (tail, small))
    if cus == 256:
        assert tail <= G.PF_SMALL_MS[-1]


@pytest.mark.gpu
def test_rounds_count_this_devices_cus(monkeypatch):
    monkeypatch.setattr(G._P, "cus", 7)
    monkeypatch.setattr(G._P, "pf_parts", {(2000, 64, 64): ((2000, (64, 64, 3, 1, 1, 4)),)})
    monkeypatch.delenv("DLLM_GEMM_PLANS", raising=False)
    G.autotune([], [], "cuda")
    assert G._P.cus == torch.cuda.get_device_properties(0).multi_processor_count and not G._P.pf_parts


def test_which_f32_products_are_taken(monkeypatch):
    monkeypatch.delenv("DLLM_GEMM", raising=False)
    rows = lambda M, K: torch.zeros(M, K)  # noqa: E731
    for M in range(1, 9):
        assert all(G.fg_takes(rows(M, K), N) for N in (16, 8192, 32000) for K in (512, 2048))
    for M, K, N, yes in [(9, 1024, 32000, True), (12, 1024, 32000, True), (13, 1024, 32000, False), (16, 1024, 16384, True), (16, 1024, 16, True),
                         (16, 2048, 128, False), (9, 2048, 8192, False), (16, 2048, 512, True), (16, 2048, 4096, True), (17, 512, 512, False)]:
        assert G.fg_takes(rows(M, K), N) == yes and G.fg_takes(rows(M, K)) == (M <= 16)
    assert not G.fg_takes(torch.zeros(4, 520)[:, 1:513], 512) and not G.fg_takes(rows(4, 512).bfloat16(), 512)


def test_prompt_parts_that_leave_most_of_a_round(monkeypatch, tmp_path):
    """TinyLlama's down product: 3487 rows behind a round of large tiles run on what was timed for the next size, also from a plan file; more than
    was timed is one launch."""
    monkeypatch.delenv("DLLM_FUSED_CORE", raising=False)
    N, K, big, tail = 2048, 5632, (256, 256, 2, 1, 1, 4), (256, 128, 3, 1, 1, 8, 1, 8)
    monkeypatch.setattr(G._P, "pf_tail", {(m, N, K): (tail, 0.02 * m) for m in G.PF_TAIL_MS})
    _none_timed(monkeypatch)
    G._P.pf_times[N, K] = [(big, 8192, 135.0)]
    G._save_plans(str(tmp_path / "plans.json"))
    _none_timed(monkeypatch)
    G._P.pf_tail.clear()
    G._load_plans(str(tmp_path / "plans.json"))
    for left, parts in ((1024, 1), (1025, 2), (1280, 2), (3487, 2), (3968, 2), (3969, 1)):
        assert len(G.prompt_parts(8192 + left, N, K)) == parts
    assert G.prompt_parts(11679, N, K) == ((8192, big), (3487, tail))
