"""Sums whose order is part of the result: what reaches an mLSTM head that divides by small sums keeps its last bit, whatever the batch
and however a launch is cut."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.models.llama import AttnMeta
from distributed_llm_amd.ops import gemm, seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"


def wave(v):
    """Sum over 64 lanes (last dim) by butterflies of 32, 16, .. 1, in f32."""
    i = torch.arange(64)
    for o in (32, 16, 8, 4, 2, 1):
        v = v + v[..., i ^ o]
    return v[..., 0]


def lanes(v, step):
    """Rows [.., n] -> per lane sums [.., step] of the squares of entries lane, lane + step, .., one after the other, in f32 (a
    square of a bf16 number is exact there)."""
    v = torch.nn.functional.pad(v, (0, -v.shape[-1] % step)).unflatten(-1, (-1, step))
    s = torch.zeros_like(v[..., 0, :])
    for j in range(v.shape[-2]):
        s = s + v[..., j, :] * v[..., j, :]
    return s


@pytest.mark.parametrize("H,groups", [(1024, 4), (1024, 1), (70, 1), (300, 1), (768, 3), (640, 5), (2048, 1), (2048, 2), (4096, 1), (4096, 2), (8192, 1), (8192, 2), (8320, 1)])
def test_norms(H, groups):
    """Each of the register forms and the general one: a workgroup on a row, a wave on a part."""
    torch.manual_seed(H)
    y, w = torch.randn(5, H).bfloat16(), torch.randn(H)
    parts = y.float().view(5, groups, -1)
    n = H // groups
    by_wave = wave(lanes(parts, 64))
    s = by_wave
    if groups == 1:
        four = wave(lanes(parts, 256).unflatten(-1, (4, 64)))
        s = ((four[..., 0] + four[..., 1]) + four[..., 2]) + four[..., 3]

    def scaled(s):
        s = s.to(DEV)      # the device's root and division (by a tensor: by a number is by its reciprocal)
        r = (1 / torch.sqrt(s / torch.full_like(s, n) + 1e-6)).cpu()
        return (parts * r[..., None]).view(5, H) * w

    x, xl = torch.zeros(5, H, device=DEV), torch.empty(5, H, device=DEV, dtype=torch.bfloat16)
    seqmix.norm_resadd(y.to(DEV), w.to(DEV), 1e-6, x, xl, groups)         # a stream of zeros: one rounding behind the product
    assert torch.equal(x.cpu(), scaled(s)) and torch.equal(xl.cpu(), scaled(s).bfloat16())
    assert torch.equal(seqmix.rms_rows(y.to(DEV), w.to(DEV), 1e-6, torch.float32, groups).cpu(), scaled(by_wave))


@pytest.mark.parametrize("T,H,groups", [(1, 64, 1), (16, 1024, 4), (5, 1088, 1), (2, 4096, 2), (3, 320, 5), (2, 8192, 2)])
def test_experts_sum(T, H, groups):
    """SwiGLU experts whose sum ends in the stream: the bits of the combine, the norm and the add one after the other."""
    torch.manual_seed(H)
    E, top = 5, 3
    x, w = torch.randn(T, H, device=DEV).bfloat16(), torch.randn(H, device=DEV)
    ids = torch.stack([torch.randperm(E, device=DEV)[:top] for _ in range(T)]).int()
    wts, st = torch.rand(T, top, device=DEV), torch.randn(T, H, device=DEV)
    w1, w2 = (torch.randn(E, a, b, device=DEV).div(b ** 0.5).bfloat16() for a, b in ((128, H), (H, 64)))
    a, b, al, bl = st.clone(), st.clone(), torch.empty_like(x), torch.empty_like(x)
    seqmix.norm_resadd(ops.moe_ffn_tg(x, ids, wts, w1, w2), w, 1e-6, a, al, groups=groups)
    assert ops.moe_ffn_tg(x, ids, wts, w1, w2, tail=(w, 1e-6, b, bl, groups)) is None
    assert torch.equal(a, b) and torch.equal(al, bl)


@pytest.mark.parametrize("N,K", [(1024, 1024), (64, 1024), (1024, 768), (5632, 1024), (1024, 2816), (4096, 1056), (1024, 4096), (2064, 64), (8192, 2048)])
def test_untimed_products(N, K):
    """A row's bits at 1 to 64 rows are those of 32 columns a workgroup and every split of K on its own."""
    torch.manual_seed(N + K)
    w = (torch.randn(N, K, device=DEV) * K ** -0.5).bfloat16()
    x = torch.randn(64, K, device=DEV).bfloat16()
    splits = gemm._heuristic(64, N, K)[2]
    want = gemm._run_plan(("skinny", 2, splits), x, w, False, None)
    assert float((want.double() - x.double() @ w.double().t()).norm() / want.double().norm()) < 2 ** -8
    for M in (1, 2, 3, 4, 8, 15, 16, 17, 24, 32, 33, 48, 63, 64):
        assert gemm._heuristic(M, N, K)[2] == splits
        assert torch.equal(ops.linear(x[:M], w), want[:M]), M
    odd = torch.randn(1, K + 4, device=DEV).bfloat16()
    odd[0, :K] = x[0]
    assert torch.equal(ops.linear(odd[:, :K], w), want[:1])           # one row of any stride


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [3, 64, 200])
def test_mamba2_prompts(dt, n):
    """A prompt in one portion and token by token: the same bits."""
    torch.manual_seed(n)
    H, dv, N, G = 4, 64, 128, 2
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    xbc, proj = torch.randn(n, H * dv + 2 * G * N, device=DEV).to(dt), torch.randn(n, H, device=DEV).to(dt)
    c = (torch.randn(H, device=DEV), -torch.rand(H, device=DEV), torch.randn(H, device=DEV))
    a, b = torch.zeros(1, H, N, dv, device=DEV), torch.zeros(1, H, N, dv, device=DEV)
    y = seqmix.ssd_scan(xbc, proj, 0, H, dv, N, G, *c, a, i32(0), i32(n), i32(n), i32(0))
    z = [seqmix.ssd_scan(xbc[t:t + 1], proj[t:t + 1], 0, H, dv, N, G, *c, b, i32(0), i32(1), i32(t + 1), i32(0)) for t in range(n)]
    assert torch.equal(y, torch.cat(z)) and torch.equal(a, b)


@pytest.mark.parametrize("lens", [[1, 1, 1], [5, 40, 130]])
def test_shared_values_f32(lens):
    """f32 maps that share their values (differential attention): the bits of the general kernel, which pages of 8 keys take."""
    torch.manual_seed(7)
    H, G, d, dv, ctxs = 8, 4, 64, 128, [n + 33 for n in lens]
    nb = [-(-c // 16) for c in ctxs]
    bt, at = torch.zeros(3, max(nb), dtype=torch.int32, device=DEV), 0
    for s, m in enumerate(nb):
        bt[s, :m] = torch.arange(at, at + m)
        at += m
    kc, vc = torch.randn(at, G, 16, d, device=DEV), torch.randn(at, G // 2, dv, 16, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    qs, ql, cx = i32([sum(lens[:s]) for s in range(3)]), i32(lens), i32(ctxs)
    q = torch.randn(sum(lens), H, d, device=DEV) * d ** -0.5
    meta = AttnMeta(slots=None, block_tables=bt, qstart=qs, qlen=ql, ctx=cx, tile_seq=None, tile_tok0=None, last_idx=None, host_qlen=lens)
    ts, tt = meta.latent_tiles(1, DEV, seqmix.gqa_tokens_per_tile(H, G, False))
    half = lambda x, keys: x.unflatten(keys, (2, 8)).movedim(keys, 1).flatten(0, 1).contiguous()  # noqa: E731
    a = seqmix.paged_gqa_attention(q, kc, vc, bt, qs, ql, cx, ts, tt, window=100)
    b = seqmix.paged_gqa_attention(q, half(kc, 2), half(vc, 3), torch.stack((2 * bt, 2 * bt + 1), 2).flatten(1).contiguous(), qs, ql, cx, ts, tt, window=100)
    assert torch.equal(a, b)
