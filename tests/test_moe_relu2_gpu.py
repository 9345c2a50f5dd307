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


def test_router_choice_of_ties_and_non_finite_logits():
    """The lower expert first among equals; NaN is never chosen; expert 0 where nothing is left to choose."""
    x = torch.zeros(4, 64, device=DEV).bfloat16()
    x[:, 0], x[1, 1], x[2, 1], x[3, 1] = 1, 1, 1, 1
    wg = torch.zeros(9, 64, device=DEV).bfloat16()
    wg[:, 0] = torch.tensor([1, 3, 2, 3, 2, 3, 0, 1, 2]).bfloat16().to(DEV)
    ids, w = ops.moe_router(x[:1], wg, 5)
    assert ids.tolist() == [[1, 3, 5, 2, 4]]
    torch.testing.assert_close(w[0].double(), torch.softmax(torch.tensor([3., 3, 3, 2, 2]).double(), 0).to(DEV), atol=1e-6, rtol=1e-6)
    bad = wg.clone()
    bad[1, 1], bad[5, 1] = float("nan"), float("-inf")
    assert ops.moe_router(x[1:2], bad, 3)[0].tolist() == [[3, 2, 4]]
    bad[:, 1] = float("-inf")
    assert ops.moe_router(x[2:3], bad, 2)[0].tolist() == [[0, 0]]


@pytest.mark.parametrize("E,top,T", [(1, 1, 1), (3, 2, 5), (64, 8, 16), (64, 8, 129), (8, 3, 700), (9, 1, 64), (40, 2, 2100)])
@pytest.mark.parametrize("pairs", [1, 600, 1 << 20])      # the plans' tiles: 64, 128 and 256 rows
def test_route_tiles(E, top, T, pairs):
    """Pairs by expert in the order of their tokens, full and partial tiles; experts without pairs, one wave and many, more pairs than a
    block: read off through experts that are multiples of the identity."""
    torch.manual_seed(E)
    H = 64
    ids = torch.stack([torch.randperm(E, device=DEV)[:top] for _ in range(T)]).int()
    ids = torch.where(ids % 5 == 2, ids // 2, ids)                      # some experts get nothing, some pairs repeat
    wts = torch.rand(T, top, device=DEV)
    x = torch.rand(T, H, device=DEV).bfloat16()
    w1 = torch.eye(H, device=DEV).expand(E, H, H).bfloat16().contiguous()
    w2 = (torch.eye(H, device=DEV)[None] * (1 + torch.arange(E, device=DEV))[:, None, None]).bfloat16()
    out = torch.empty(T, H, device=DEV).bfloat16()
    ops._native(x).moe_ffn_tg(x, ids, wts, w1, w2, out, list(ops.moe_plan(pairs)), 1)
    want = (x.double() ** 2) * ((ids + 1).double() * wts.double()).sum(1, keepdim=True)
    assert float((out.double() - want).norm() / want.norm()) < 2 ** -8


@pytest.mark.parametrize("T,H,groups", [(1, 64, 1), (24, 1024, 4), (5, 1088, 1), (3, 2048, 8), (2, 4096, 16), (2, 8192, 2), (7, 320, 5), (2, 8256, 1)])
@pytest.mark.parametrize("mode", [0, 1])
def test_tail(T, H, groups, mode):
    """The weighted sum, its norm and the residual add in one launch, and on widths that take their own launches (parts that are no whole
    256s, rows past 8192)."""
    torch.manual_seed(H)
    E, top, I = 5, 3, 64
    x = torch.randn(T, H, device=DEV).bfloat16()
    ids = torch.stack([torch.randperm(E, device=DEV)[:top] for _ in range(T)]).int()
    wts, w, st = torch.rand(T, top, device=DEV), torch.randn(H, device=DEV), torch.randn(T, H, device=DEV)
    w1, w2 = (torch.randn(E, a, b, device=DEV).div(b ** 0.5).bfloat16() for a, b in (((2 - mode) * I, H), (H, I)))
    run = (lambda **kw: ops.moe_ffn_tg(x, ids, wts, w1, w2, **kw)) if mode == 0 else (lambda **kw: seqmix.moe_ffn_relu2(x, ids, wts, w1, w2, **kw))
    y = run().double()
    want = st.double() + (y.view(T, groups, -1) * torch.rsqrt(y.view(T, groups, -1).pow(2).mean(-1, keepdim=True) + 1e-6)).view(T, H) * w.double()
    s2, xl = st.clone(), torch.empty_like(x)
    assert run(tail=(w, 1e-6, s2, xl, groups)) is None
    # y above was rounded to bf16 (2^-9 an element); the stream is f32
    assert float((s2.double() - want).norm() / want.norm()) < 2 ** -8
    assert torch.equal(xl, s2.bfloat16())
    s3 = st.clone()
    assert run(tail=(w, 1e-6, s3, None, groups)) is None
    assert torch.equal(s2, s3)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H,groups,pad", [(3, 1024, 4, 0), (2, 1020, 1, 4), (5, 64, 1, 0), (2, 2304, 9, 8), (1, 8192, 1, 0), (2, 6144, 3, 0), (2, 768, 6, 0), (3, 70, 1, 1)])
@pytest.mark.parametrize("bias", [False, True])
def test_norm_resadd_widths(dt, T, H, groups, pad, bias):
    """Rows in registers: 1 to 8 vectors a thread, rows that fill no workgroup, parts of whole 256s; other widths take the general form."""
    torch.manual_seed(H)
    y = torch.randn(T, H + pad, device=DEV).to(dt)[:, :H]
    w, x, b = torch.randn(H, device=DEV), torch.randn(T, H, device=DEV), torch.randn(H, device=DEV) if bias else None
    z = y.double() + (b.double() if bias else 0)
    want = x.double() + (z.view(T, groups, -1) * torch.rsqrt(z.view(T, groups, -1).pow(2).mean(-1, keepdim=True) + 1e-5)).view(T, H) * w.double()
    xl = torch.empty(T, H, device=DEV, dtype=dt)
    seqmix.norm_resadd(y, w, 1e-5, x, xl, groups, b)
    assert float((x.double() - want).norm() / want.norm()) < 1e-6
    assert torch.equal(xl, x.to(dt))


@pytest.mark.parametrize("T,H", [(1, 64), (16, 1024), (5, 1032), (3, 2048), (2, 4096), (2, 8192)])
@pytest.mark.parametrize("n,E,top,count,keep,score,gscore,real", [(8, 8, 2, 2, 1, "sigmoid", "top2", 8), (13, 12, 3, 4, 2, "softmax", "max", 10),
                                                                  (256, 256, 8, 8, 4, "sigmoid", "top2", 256), (1, 1, 1, 1, 1, "softmax", "top2", 1)])
def test_router_topk(T, H, n, E, top, count, keep, score, gscore, real):
    """Logits, choice and weights of the one launch against f64 logits through the standalone routing; 1 to 16 vectors a lane, outputs
    that fill no round of the waves, a column behind the routed ones."""
    torch.manual_seed(n + H)
    x = torch.randn(T, H + 8, device=DEV).bfloat16()[:, :H]
    w, corr = torch.randn(n, H, device=DEV) / H ** 0.5, torch.randn(E, device=DEV) * 0.1
    ids, wt, idw, lg = seqmix.router_topk(x, w, E, top, count, keep, score, gscore, corr, real, want_logits=True)
    want = x.double() @ w.double().t()
    assert float((lg.double() - want).abs().max()) < 2e-5          # H products of order H^-1/2 summed in f32
    i2, w2, d2 = seqmix.route_topk(lg, E, top, count, keep, score, gscore, corr, real)
    assert torch.equal(ids, i2) and torch.equal(wt, w2) and torch.equal(idw, d2)
    i3, w3, d3, none = seqmix.router_topk(x, w, E, top, count, keep, score, gscore, corr, real)
    assert none is None and torch.equal(ids, i3) and torch.equal(wt, w3) and torch.equal(idw, d3)
    one = seqmix.router_topk(x[-1:], w, E, top, count, keep, score, gscore, corr, real, want_logits=True)
    assert torch.equal(one[3], lg[-1:])                            # a token's logits do not depend on the batch


@pytest.mark.parametrize("T,H,E,top", [(1, 64, 4, 2), (12, 1024, 8, 2), (5, 1088, 8, 1), (9, 2048, 64, 8), (3, 4096, 8, 2), (2, 8192, 5, 3), (700, 512, 8, 2)])
def test_norm_router_and_residual_combine(T, H, E, top):
    """Norm + router and combine + residual add against the launches they replace: 1 to 16 vectors a lane, one and several slots."""
    torch.manual_seed(H)
    r = torch.randn(T, H + 8, device=DEV).bfloat16()[:, :H]
    nw, wg = torch.randn(H, device=DEV).bfloat16(), torch.randn(E, H, device=DEV).bfloat16()
    x, ids, w = ops.norm_moe_router(r, nw, 1e-5, wg, top)
    z = r.double() * torch.rsqrt(r.double().pow(2).mean(-1, keepdim=True) + 1e-5) * nw.double()
    assert float((x.double() - z).norm() / z.norm()) < 2 ** -8          # one rounding to bf16
    i2, w2 = ops.moe_router(x, wg, top)
    assert torch.equal(ids, i2) and torch.equal(w, w2)                   # the rounded rows are what is routed
    w13, w2d = torch.randn(E, 128, H, device=DEV).div(H ** 0.5).bfloat16(), torch.randn(E, H, 64, device=DEV).div(8).bfloat16()
    for slots in (1, 3):
        ra, rb = r.clone(), r.clone()
        qa, qb = (torch.zeros(slots, T + 2, device=DEV) for _ in range(2))
        na = ops.moe_ffn_tg_resadd(x, ids, w, w13, w2d, ra, qa)
        nb = ops.gemm.res_add_ssq(ops.moe_ffn_tg(x, ids, w, w13, w2d), rb, qb)
        assert na == nb and torch.equal(ra, rb) and torch.equal(qa, qb)


@pytest.mark.parametrize("ti", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("to", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,n,groups,pad", [(24, 1024, 1, 0), (5, 256, 1, 8), (3, 260, 1, 4), (7, 4, 1, 0), (2, 4096, 1, 0), (2, 4100, 1, 0), (3, 2048, 4, 0), (3, 70, 1, 0),
                                            (3, 768, 3, 1), (1, 1536, 1, 0)])
@pytest.mark.parametrize("weight", [False, True])
def test_rms_rows_widths(ti, to, T, n, groups, pad, weight):
    """Parts in registers: 1 to 16 vectors a lane, full and not; unaligned rows, odd widths and parts past 4096 take the other form."""
    torch.manual_seed(n)
    x = torch.randn(T, n + pad, device=DEV).to(ti)[:, :n]
    w = torch.randn(n, device=DEV) if weight else None
    z = x.double().reshape(T, groups, -1)
    want = (z * torch.rsqrt(z.pow(2).mean(-1, keepdim=True) + 1e-6)).reshape(T, n) * (w.double() if weight else 1)
    got = seqmix.rms_rows(x, w, 1e-6, to, groups)
    # one rounding to the output's type (f32: the sum's and the root's few units of 2^-24 beside it)
    assert float((got.double() - want).norm() / want.norm()) < (1e-6 if to == torch.float32 else 2 ** -9)
