"""The 256 x 256 tile of four waves (csrc/kernels/wide_gemm.hip) against the 64 x 64 tile: a product's terms are added in the same order, so the
results are the same bits, at the edges of its tiles and of its ring (one, two and three 64-deep stages)."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import gemm as G

pytestmark = pytest.mark.gpu
WIDE, SMALL = (256, 256, 2, 1, 1, 4), (64, 64, 3, 1, 1, 4)
RASTER = WIDE + (1, 0, 0, 64, 16, 8)
SIZES = [(1, 256, 64), (255, 64, 128), (256, 256, 192), (257, 320, 320), (300, 40, 64), (2600, 544, 128), (513, 1056, 2048)]


def rnd(*s, scale=1.0):
    return (torch.randn(*s, device="cuda") * scale).to(torch.bfloat16)


def ext():
    return ops._load()


def both(run, plans=(SMALL, WIDE, RASTER)):
    got = [run(p) for p in plans]
    assert all(torch.equal(a, b) for g in got[1:] for a, b in zip(g, got[0]))
    return got[0]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("panel", [False, True])
def test_plain_and_bias(M, N, K, panel):
    torch.manual_seed(M)
    x, w, b = rnd(M, K + 8)[:, :K], rnd(N, K, scale=0.05), rnd(N)
    if panel and N % 64:
        pytest.skip("panel copies have whole 64-row tiles")
    wk = G.panel_weight(w) if panel else w

    def run(epi, bias):
        def f(p):
            y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
            G._tgemm(ext(), x, wk, epi, p, y=y, bias=bias)
            return (y,)
        return f
    y, = both(run(G.EPI_PLAIN, None))
    want = x.double() @ w.double().t()
    # the f32 sums of K products, then one rounding to 8 bits
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -22 * x.abs().double() @ w.abs().double().t()).all()
    if not panel:
        both(run(G.EPI_PLAIN, b))
        both(run(G.EPI_GELU, b))


@pytest.mark.parametrize("M,N,K", SIZES)
def test_residual(M, N, K):
    torch.manual_seed(M)
    x, w, r = rnd(M, K), rnd(N, K, scale=0.05), rnd(M, N)

    def run(p):
        y, ssq = r.clone(), torch.zeros(G.max_slots(N), M, device="cuda")
        G._tgemm(ext(), x, w, G.EPI_RESADD, p, y=y, ssq_out=ssq)
        # (f32 sums of N squares in another order)
        torch.testing.assert_close(ssq.double().sum(0), (y.double() ** 2).sum(1), rtol=N * 2.0 ** -24, atol=0)
        return (y,)
    both(run)


@pytest.mark.parametrize("M,N,K", [(1, 64, 64), (257, 544, 192), (700, 2048, 128)])
@pytest.mark.parametrize("slots", [0, 1, 19])
def test_swiglu(M, N, K, slots):
    torch.manual_seed(M)
    x, w, ssq = rnd(M, K), rnd(N, K, scale=0.05), torch.rand(max(1, slots), M, device="cuda") + 0.5
    ssq = torch.floor(ssq * 64) / 64      # (sums of multiples of 1 / 64: the same in any order)

    def run(p):
        y = torch.full((M, N // 2), float("nan"), dtype=torch.bfloat16, device="cuda")
        kw = dict(ssq_in=ssq, ssq_n=slots, norm_scale=1.0 / 16, eps=1e-5) if slots else {}
        G._tgemm(ext(), x, w, G.EPI_SWIGLU, p, y=y, **kw)
        return (y,)
    both(run)


@pytest.mark.parametrize("M,d,nq,nkv,v_rows", [(1, 64, 8, 2, False), (256, 64, 32, 4, True), (300, 96, 3, 1, False), (515, 128, 4, 4, False)])
def test_qkv(M, d, nq, nkv, v_rows):
    torch.manual_seed(M)
    K, blocks = 192, 64
    N = (nq + 2 * nkv) * d
    x, w = rnd(M, K), rnd(N, K, scale=0.05)
    ssq, cos_sin = torch.rand(1, M, device="cuda") * K, torch.rand(4096, d, device="cuda")
    pos = torch.randint(0, 4096, (M,), device="cuda", dtype=torch.int32)
    slots = torch.arange(3, M + 3, device="cuda", dtype=torch.int32)      # runs of eight slots that start inside the tile
    slots[::7] = -1

    def run(p):
        q = torch.zeros(M, nq, d, dtype=torch.bfloat16, device="cuda")
        kc, vc = (torch.zeros(blocks, nkv, *s, dtype=torch.bfloat16, device="cuda") for s in ((16, d), (d, 16)))
        v = torch.zeros(M, nkv * d, dtype=torch.bfloat16, device="cuda") if v_rows else None
        G._tgemm(ext(), x, w, G.EPI_QKV, p, ssq_in=ssq, ssq_n=1, norm_scale=1.0 / K, eps=1e-5, pos=pos, cos_sin=cos_sin, slots=slots,
                 q_out=q, kc=kc, vc=vc, nq=nq, nkv=nkv, d=d, v_rows=v)
        return (q, kc, vc) + ((v,) if v_rows else ())
    both(run)


@pytest.mark.parametrize("relu2", [False, True])
@pytest.mark.parametrize("T,E,k,H,I", [(1, 2, 1, 64, 128), (300, 3, 2, 320, 192), (2000, 5, 3, 256, 576)])
def test_experts(T, E, k, H, I, relu2):
    """Ragged row tiles of the grouped form, one expert without rows; both products, gathered and in place."""
    torch.manual_seed(T)
    x, ids = rnd(T, H), torch.stack([torch.randperm(E - 1, device="cuda")[:k] for _ in range(T)]).int()
    wts = torch.rand(T, ids.shape[1], device="cuda")
    w1, w2 = rnd(E, I if relu2 else 2 * I, H, scale=0.05), rnd(E, H, I, scale=0.05)

    def run(p):
        return (ops.moe_run_tg(ext(), x, ids, wts, w1, w2, p, int(relu2), None),)
    both(run, ((256, 128, 3, 1, 8, 128, 3, 1, 8), (256, 256, 2, 1, 4, 128, 3, 1, 8), (256, 256, 2, 1, 4, 256, 2, 1, 4)))


def test_refused():
    """More than one split and other depths have no such tile."""
    x, w, y = rnd(64, 512), rnd(256, 512), torch.empty(64, 256, dtype=torch.bfloat16, device="cuda")
    for p in ((256, 256, 2, 2, 1, 4), (256, 256, 2, 1, 2, 4), (256, 256, 3, 1, 1, 4), (256, 128, 2, 1, 1, 4)):
        with pytest.raises(RuntimeError):
            G._tgemm(ext(), x, w, G.EPI_PLAIN, p, y=y)
