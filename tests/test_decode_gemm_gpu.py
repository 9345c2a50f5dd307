"""Decode GEMM on fragment-major weights (csrc/kernels/decode_gemm.hip): every epilogue at edges of the row and column tiles, tails of K
and splits over waves, groups and workgroups."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.models.llama import fuse_gate_up_weight, fuse_qkv_weight
from distributed_llm_amd.ops import gemm as G
from distributed_llm_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROWS = [1, 5, 16, 17, 32, 33, 48, 49, 64]
# (16-column tiles, splits a workgroup, splits): all in a workgroup, apart, both, a group without k
PLANS = [(1, 1, 1), (2, 1, 3), (3, 1, 1), (1, 2, 2), (2, 2, 4), (3, 2, 2), (2, 2, 3), (1, 2, 1)]


def _rnd(*s, scale=1.0):
    return (torch.randn(*s, device=DEV) * scale).bfloat16()


def _close(got, want, K):
    """f32 sums of K products in another order, then one bf16 rounding."""
    err = (got.float() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 1e-6 * K * want.abs().max()).all(), err.max()


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("plan", PLANS + [(1, 4, 4), (1, 4, 3)])
@pytest.mark.parametrize("N,K", [(96, 32), (90, 416), (1024, 1024), (272, 2816)])
def test_plain(M, plan, N, K):
    nt, vs, sp = plan
    if vs == 4 and M > 32:
        pytest.skip("four splits a workgroup: up to 32 rows")
    torch.manual_seed(M + N)
    G.reserve(DEV)
    x, w = _rnd(M, K + 8)[:, :K], _rnd(N, K, scale=0.05)
    y = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    wf = G.frag_weight(w)
    for _ in range(2):      # tickets are armed again
        G.dgemm(x, wf, N, G.EPI_PLAIN, plan, y=y)
    _close(y, (x.double() @ w.double().t()).float(), K)
    if nt < 3:      # the row-major kernel with as many splits: the same bits, however the launch is cut
        s = torch.empty_like(y)
        floats, tiles = G._need(M, N, K, nt, sp)
        part, cnt = G._P.workspace(x.device, floats, tiles)
        G._native(x).skinny_gemm(x, w, s, nt, sp, False, part, cnt, 1)
        assert torch.equal(s, y)


@pytest.mark.parametrize("M", [1, 4, 24, 48, 64])
@pytest.mark.parametrize("N,K", [(1024, 1024), (4096, 1024), (3088, 1024), (1024, 4096), (128, 2048), (5632, 1024)])
def test_untimed_products_keep_their_bits(M, N, K):
    x, w = _rnd(M, K), _rnd(N, K, scale=0.05)
    assert torch.equal(G.linear(x, w), G.linear(x, w, wf=G.frag_weight(w)))


def test_rows_do_not_meet():
    """A row's infinities and NaN stay in it."""
    x, w = _rnd(40, 512), _rnd(64, 512)
    want = torch.empty(40, 64, dtype=torch.bfloat16, device=DEV)
    got = torch.empty_like(want)
    G.dgemm(x, G.frag_weight(w), 64, G.EPI_PLAIN, (1, 2, 2), y=want)
    x[7, 100], x[20, 3] = float("nan"), float("inf")
    G.dgemm(x, G.frag_weight(w), 64, G.EPI_PLAIN, (1, 2, 2), y=got)
    keep = [i for i in range(40) if i not in (7, 20)]
    assert torch.equal(got[keep], want[keep]) and got[7].isnan().all() and not got[20].isfinite().any()


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("N,K", [(256, 512), (2048, 2048), (100, 5632)])
def test_resadd(M, plan, N, K):
    torch.manual_seed(M * 7 + N)
    G.reserve(DEV)
    x, w, r = _rnd(M, K), _rnd(N, K, scale=0.02), _rnd(M, N)
    r0, ssq = r.clone(), torch.full((G.max_slots(N, M), M), float("nan"), device=DEV)
    n = G.dgemm(x, G.frag_weight(w), N, G.EPI_RESADD, plan, res=r, ssq_out=ssq)
    assert n == -(-N // (16 * plan[0]))
    want = (x.double() @ w.double().t()).float()
    # the product's and the sum's bf16 roundings
    err = (r.float() - (want + r0.float())).abs()
    assert (err <= 2.0 ** -7 * (want.abs() + r0.float().abs()) + 1e-6 * K * want.abs().max()).all(), err.max()
    torch.testing.assert_close(ssq[:n].sum(0), (r.float() ** 2).sum(1), rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("v_rows", [False, True])
@pytest.mark.parametrize("d,nq,nkv,H", [(64, 8, 2, 256), (32, 4, 1, 512), (128, 32, 8, 4096), (96, 4, 2, 320)])
def test_qkv(M, plan, v_rows, d, nq, nkv, H):
    torch.manual_seed(M + d)
    G.reserve(DEV)
    r, ln = _rnd(M, H), (1.0 + 0.1 * torch.randn(H, device=DEV)).bfloat16()
    wqkv = _rnd((nq + 2 * nkv) * d, H, scale=0.05)
    wf = G.frag_weight(fuse_qkv_weight(wqkv, ln, nq, nkv, d), paired=True)
    cs = ops.rope_cos_sin(4096, d, 10000.0, DEV)
    pos = torch.randint(0, 4000, (M,), device=DEV, dtype=torch.int32)
    slots = torch.randperm(96, device=DEV)[:M].to(torch.int32)
    if M > 2:
        slots[1] = -1
    kc = torch.zeros(6, nkv, 16, d, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros(6, nkv, d, 16, dtype=torch.bfloat16, device=DEV)
    q = torch.empty(M, nq, d, dtype=torch.bfloat16, device=DEV)
    vn = torch.empty(M, nkv * d, dtype=torch.bfloat16, device=DEV) if v_rows else None
    G.dgemm(r, wf, (nq + 2 * nkv) * d, G.EPI_QKV, plan, scale=1.0 / H, eps=1e-5, pos=pos, cos_sin=cs, slots=slots, q_out=q, kc=kc, vc=vc,
            v_rows=vn, nq=nq, nkv=nkv, d=d)
    qkv = (ref.rms_norm(r.cpu(), ln.cpu(), 1e-5).float() @ wqkv.cpu().float().t()).bfloat16()
    kr, vr = torch.zeros(6, nkv, 16, d, dtype=torch.bfloat16), torch.zeros(6, nkv, d, 16, dtype=torch.bfloat16)
    qr = ref.rope_and_cache(qkv, pos.cpu(), cs.cpu(), slots.cpu(), kr, vr, nq, nkv, d)
    # norm weight folded into bf16 columns, a rounding ahead of the rotation: 2^-8 of sums of H terms of 0.05 each, and of the pair
    tol = 2.0 ** -6 * qkv.float().abs().max().item()
    torch.testing.assert_close(q.cpu().float(), qr.float(), atol=tol, rtol=2e-2)
    torch.testing.assert_close(kc.cpu().float(), kr.float(), atol=tol, rtol=2e-2)
    if v_rows:
        torch.testing.assert_close(vn.cpu().float(), qkv[:, (nq + nkv) * d:].float(), atol=tol, rtol=2e-2)
        assert not vc.any()
    else:
        torch.testing.assert_close(vc.cpu().float(), vr.float(), atol=tol, rtol=2e-2)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("H,I", [(256, 320), (2048, 5632), (96, 16)])
def test_swiglu(M, plan, H, I):
    torch.manual_seed(M + I)
    G.reserve(DEV)
    r, ln = _rnd(M, H), (1.0 + 0.1 * torch.randn(H, device=DEV)).bfloat16()
    wgu = _rnd(2 * I, H, scale=0.05)
    act = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
    G.dgemm(r, G.frag_weight(fuse_gate_up_weight(wgu, ln), paired=True), 2 * I, G.EPI_SWIGLU, plan, y=act, scale=1.0 / H, eps=1e-5)
    gu = (ref.rms_norm(r.cpu(), ln.cpu(), 1e-5).float() @ wgu.cpu().float().t()).bfloat16()
    want = ref.silu_mul(gu).float()
    # each factor to 2^-6 of the largest (as test_qkv), the product of two
    torch.testing.assert_close(act.cpu().float(), want, atol=2.0 ** -6 * gu.float().abs().max().item() * 2, rtol=2e-2)


@pytest.mark.parametrize("M", [1, 4, 17, 48, 64])
@pytest.mark.parametrize("act,limit,alpha,bias", [("gelu", 0.0, 1.0, False), ("swiglu", 0.0, 1.0, False), ("clamped", 1.5, 1.702, True),
                                                  ("gelu_tanh", 0.0, 1.0, True), ("gelu_tanh", 0.0, 1.0, False)])
@pytest.mark.parametrize("N,K", [(5632, 1024), (4096, 1024), (144, 96), (1024, 4096)])
def test_activations(M, act, limit, alpha, bias, N, K):
    """The activation in the product's launch: the bits of the two launches."""
    from distributed_llm_amd.ops import seqmix
    torch.manual_seed(M + N)
    G.reserve(DEV)
    x, w = _rnd(M, K), _rnd(N, K, scale=2 * K ** -0.5)
    b = torch.randn(N, device=DEV) if bias else None
    got = G.linear_act(x, w, G.frag_weight(w, paired=False if act == "gelu" else "glu"), act, b, limit, alpha)
    z = G.linear(x, w, wf=G.frag_weight(w))
    want = seqmix.gelu_erf(z) if act == "gelu" else seqmix.glu_act(z, b, act, limit, alpha)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M", [1, 2, 15, 16])
@pytest.mark.parametrize("N,K", [(16, 16), (90, 48), (515, 512), (1000, 1040), (256, 2048)])
def test_f32_rows(M, N, K):
    """The f32 product: waves without a step, partial groups of steps, columns past N, rows of a wider matrix; against a double's.  A sum is
    at most K / 8 + 15 terms in a row and eight of those: that many roundings of 2^-24 of the absolute sum; erf-GELU (slope at most
    1.13) adds four of its own of a value or of 1."""
    x, w = torch.randn(M, K + 4, device=DEV)[:, :K], torch.randn(N, K, device=DEV)
    assert G.fg_takes(x) and not G.fg_takes(torch.randn(17, K, device=DEV)) and not G.fg_takes(torch.randn(M + 1, K + 1, device=DEV)[:, 1:])
    want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    wf = G.frag_weight(w)
    err = (G.f32_linear(x, wf, N).double() - want).abs()
    bound = (K / 8 + 24) * 2.0 ** -24 * size
    assert (err <= bound).all()
    got = G.f32_linear(x, wf, N, gelu=True).double()
    assert ((got - torch.nn.functional.gelu(want)).abs() <= 1.13 * bound + 4 * 2.0 ** -24 * (want.abs() + 1)).all()


@pytest.mark.parametrize("plan", [(1, 1, 1), (3, 1, 1), (1, 2, 2), (1, 4, 4), (2, 2, 3), (1, 4, 3)])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 17])
def test_stages_of_a_wave(plan, steps):
    """One to three half stages have a form each, longer waves walk: on both sides of every line, with whole steps for all four waves of a
    group, one more and one less."""
    for M in (4, 24):
        for K in (128 * steps * plan[2], 128 * steps * plan[2] + 32, 128 * steps * plan[2] - 32):
            test_plain(M, plan, 48, K)
