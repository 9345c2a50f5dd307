"""Router encoder on HIP (csrc/kernels/encoder.hip + tgemm bias/GELU/residual epilogues) against
fp32 PyTorch references: bidirectional attention with padding masks, fused embedding+LayerNorm,
bias GEMMs, and the whole MiniLM forward (random weights and biases; real all-MiniLM-L6-v2
weights are not fetchable here, so semantic parity with the reference stays unpinned)."""
import math

import pytest
import torch
import torch.nn.functional as F

from distributed_llm_amd import ops
from distributed_llm_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _b(*s, scale=1.0):
    return (torch.randn(*s, device="cuda") * scale).to(torch.bfloat16)


@pytest.mark.parametrize("B,S,nh,d", [(5, 77, 12, 32), (3, 512, 12, 32), (4, 40, 6, 64), (1, 1, 12, 32),
                                      (7, 33, 12, 32)])
def test_encoder_attention_matches_fp32(B, S, nh, d):
    torch.manual_seed(B * S + d)
    qkv = _b(B * S, 3 * nh * d)
    lens = torch.randint(1, S + 1, (B,), dtype=torch.int32)
    lens[0] = S
    got = ops.encoder_attention(qkv, lens.cuda(), B, S, nh, d)
    want = ref.encoder_attention(qkv.cpu(), lens, B, S, nh, d, 1.0 / math.sqrt(d))
    assert torch.isfinite(got.float()).all()
    torch.testing.assert_close(got.cpu().float(), want.float(), atol=2e-2, rtol=2e-2)


def test_embed_ln_matches_fp32():
    torch.manual_seed(3)
    V, P, H, B, S = 1000, 512, 384, 6, 21
    word, pos, type0 = _b(V, H, scale=0.5), _b(P, H, scale=0.5), _b(H, scale=0.5)
    w, b = _b(H, scale=0.3) + 1, _b(H, scale=0.3)
    ids = torch.randint(0, V, (B, S), dtype=torch.int32)
    got = ops.embed_ln(ids.cuda(), word, pos, type0, w, b, S, 1e-12)
    want = ref.embed_ln(ids, word.cpu(), pos.cpu(), type0.cpu(), w.cpu(), b.cpu(), S, 1e-12)
    torch.testing.assert_close(got.cpu().float(), want.float(), atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("M", [1, 37, 300, 1281])
@pytest.mark.parametrize("N,K", [(1152, 384), (1536, 384), (384, 1536)])
def test_bias_gemm_epilogues(M, N, K):
    torch.manual_seed(M + N)
    x, w, bias = _b(M, K), _b(N, K, scale=0.05), _b(N, scale=0.5)
    y = ops.gemm.linear_bias(x, w, bias)
    lin = x.cpu().float() @ w.cpu().float().t() + bias.cpu().float()
    torch.testing.assert_close(y.cpu().float(), lin, atol=3e-2, rtol=2e-2)
    g = ops.gemm.linear_bias(x, w, bias, gelu=True)
    torch.testing.assert_close(g.cpu().float(), F.gelu(lin.to(torch.bfloat16).float()), atol=3e-2, rtol=2e-2)
    r = _b(M, N)
    r0 = r.cpu().float()
    ops.gemm.linear_bias_residual(x, w, bias, r)
    torch.testing.assert_close(r.cpu().float(), lin.to(torch.bfloat16).float() + r0, atol=6e-2, rtol=2e-2)


def test_minilm_forward_matches_fp32_reference():
    from distributed_llm_amd.models.minilm import MiniLMEncoder
    enc = MiniLMEncoder(device="cuda", memo_size=0)
    g = torch.Generator().manual_seed(0)
    rb = lambda t, s: (torch.randn(t.shape, generator=g) * s).to(t.device, t.dtype)
    enc.emb_ln = (enc.emb_ln[0] + rb(enc.emb_ln[0], 0.1), rb(enc.emb_ln[1], 0.1))
    for L in enc.layers:   # non-zero biases and LayerNorm affine params exercise every epilogue
        for k in ("bqkv", "bo", "b1", "b2"):
            L[k] = rb(L[k], 0.05)
        for k in ("ln1", "ln2"):
            L[k] = (L[k][0] + rb(L[k][0], 0.1), rb(L[k][1], 0.1))
    texts = ["How do I reverse a linked list in Python?", "hi", "Explain the theory of relativity " * 12,
             "Write a SQL query joining orders and customers, then explain the plan", "?"]
    got = enc.encode(texts)
    want = enc.reference_forward(texts)
    cos = (got.cpu().float() * want).sum(-1)
    assert cos.min().item() > 0.999, cos
    assert enc.memo_stats()["encoded_texts"] == len(texts)


@pytest.mark.parametrize("lens", [[1], [16], [77, 1, 32, 33, 64, 65, 2], [512, 3], [5] * 40])
@pytest.mark.parametrize("nh,d", [(12, 32), (3, 64), (5, 32)])
def test_packed_batch(lens, nh, d):
    """Rows one behind the other: attention, embedding positions and pooling against each text on its own; texts that end at and past
    the kernels' blocks of 32 keys and 64 queries, widths with one and several row groups."""
    torch.manual_seed(len(lens) + d)
    H, T, S = nh * d, sum(lens), max(lens)
    starts = [sum(lens[:i]) for i in range(len(lens))]
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    qkv = _b(T, 3 * H)
    got = ops.encoder_attention(qkv, dev(lens), len(lens), S, nh, d, starts=dev(starts))
    word, pos, t0, w, b = _b(100, H, scale=0.5), _b(512, H, scale=0.5), _b(H, scale=0.5), _b(H, scale=0.3) + 1, _b(H, scale=0.3)
    ids, at = torch.randint(0, 100, (T,), dtype=torch.int32), [p for n in lens for p in range(n)]
    emb = ops.embed_ln(ids.cuda(), word, pos, t0, w, b, S, 1e-12, dev(at))
    pool = ops.mean_pool_l2(emb, dev(lens), dev(starts))
    for i, (a, n) in enumerate(zip(starts, lens)):
        one = torch.tensor([n], dtype=torch.int32).cuda()
        # the same arithmetic row by row: a padded batch of one text gives the same bits
        assert torch.equal(got[a:a + n], ops.encoder_attention(qkv[a:a + n].contiguous(), one, 1, n, nh, d))
        assert torch.equal(emb[a:a + n], ops.embed_ln(ids[None, a:a + n].cuda(), word, pos, t0, w, b, n, 1e-12))
        want = F.normalize(emb[a:a + n].double().mean(0), dim=0)
        # n rows summed in f32: n roundings of 2^-24 at most, far below
        assert float((pool[i].double() - want).norm()) < 1e-6


@pytest.mark.parametrize("H", [4, 8, 100, 384, 1000, 1024, 2048])
def test_mean_pool_widths(H):
    x = _b(3, 9, H)
    lens = torch.tensor([9, 1, 6], dtype=torch.int32).cuda()
    got = ops.mean_pool_l2(x, lens)
    for i, n in enumerate(lens.tolist()):
        assert float((got[i].double() - F.normalize(x[i, :n].double().mean(0), dim=0)).norm()) < 1e-6


@pytest.mark.parametrize("lens", [[16], [3] * 30, [70, 30, 5, 64] * 8])
@pytest.mark.parametrize("nh,d,inter", [(12, 32, 1536), (4, 64, 512), (2, 32, 96), (3, 32, 256)])
def test_layers_in_one_call(lens, nh, d, inter):
    """The same launches with the same plans as one call per operation (widths that are no multiple of 64 take those): equal bits."""
    torch.manual_seed(inter)
    H, T, S = nh * d, sum(lens), max(lens)
    layers = [dict(wqkv=_b(3 * H, H, scale=0.05), bqkv=_b(3 * H), wo=_b(H, H, scale=0.05), bo=_b(H), ln1=(_b(H) + 1, _b(H)), w1=_b(inter, H, scale=0.05),
                   b1=_b(inter), w2=_b(H, inter, scale=0.05), b2=_b(H), ln2=(_b(H) + 1, _b(H))) for _ in range(2)]
    x0 = _b(T, H)
    dl = torch.tensor(lens, dtype=torch.int32).cuda()
    ds = torch.tensor([sum(lens[:i]) for i in range(len(lens))], dtype=torch.int32).cuda()
    got = ops.gemm.encoder_layers(x0.clone(), dl, ds, S, nh, d, 1e-12, layers)
    x = x0.clone()
    for L in layers:
        a = ops.encoder_attention(ops.gemm.linear_bias(x, L["wqkv"], L["bqkv"]), dl, len(lens), S, nh, d, starts=ds)
        x = ops.layer_norm(ops.gemm.linear_bias_residual(a, L["wo"], L["bo"], x), *L["ln1"], 1e-12)
        f = ops.gemm.linear_bias(x, L["w1"], L["b1"], gelu=True)
        x = ops.layer_norm(ops.gemm.linear_bias_residual(f, L["w2"], L["b2"], x), *L["ln2"], 1e-12)
    assert torch.equal(got, x)


@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 48, 63, 64])
@pytest.mark.parametrize("N,K", [(16, 64), (48, 384), (1152, 320), (384, 1536), (64, 832), (32, 768)])
def test_few_row_projections(M, N, K):
    """Blocks of 16 rows full and not, waves without a step of K, partial groups of three steps, rows of a wider matrix."""
    torch.manual_seed(M + N)
    x, w, bias, y0 = _b(M, K + 8)[:, :K], _b(N, K, scale=K ** -0.5), _b(N, scale=0.5), _b(M, N)
    ext = ops._native(x)
    z = (x.double() @ w.double().t() + bias.double())
    for epi, want in ((0, z), (1, z + y0.double()), (4, F.gelu(z))):
        y = y0.clone()
        assert ext.enc_gemm(x, w, bias, y, epi)
        # two roundings to bf16 of at most 2^-9 each (the projection and the result)
        assert float((y.double() - want).norm() / want.norm()) < 2 ** -8
    assert not ext.enc_gemm(_b(65, K), w, bias, _b(65, N), 0) and not ext.enc_gemm(x, _b(N + 8, K), _b(N + 8), _b(M, N + 8), 0)


@pytest.mark.parametrize("M", [3, 16, 40, 64])
@pytest.mark.parametrize("K", [128, 256, 448, 512, 896, 1024, 1280, 2048, 3072, 4096])
def test_k_steps_at_a_time(M, K):
    """Two, three and four k-steps of a wave at a time."""
    test_few_row_projections(M, 48, K)


@pytest.mark.parametrize("lens", [[1], [15], [16], [17], [9, 7], [1] * 16, [1, 0, 12]])
@pytest.mark.parametrize("nh,d,inter", [(12, 32, 1536), (6, 64, 320), (3, 64, 96), (1, 32, 32), (5, 32, 64), (3, 64, 128), (2, 32, 64), (10, 32, 704),
                                        (1, 64, 64)])      # (widths that are no whole 64s take one launch an operation)
def test_layers_of_few_rows(lens, nh, d, inter):
    """Four launches a layer against one per operation.  A single text meets the same sums in the same order: equal bits.
    Among several, a text's keys lie in other lanes and its sums take another order: rows then lie no further from a
    double's than the separate launches' do, give or take a tenth (root mean square over at least 416 numbers; most of either error is
    the roundings both share)."""
    torch.manual_seed(sum(lens) + inter)
    H, T, S = nh * d, sum(lens), max(lens)
    layers = [dict(wqkv=_b(3 * H, H, scale=0.05), bqkv=_b(3 * H), wo=_b(H, H, scale=0.05), bo=_b(H), ln1=(_b(H) + 1, _b(H)), w1=_b(inter, H, scale=0.05),
                   b1=_b(inter), w2=_b(H, inter, scale=0.05), b2=_b(H), ln2=(_b(H) + 1, _b(H))) for _ in range(2)]
    x0 = _b(T, H)
    starts = [sum(lens[:i]) for i in range(len(lens))]
    dl, ds = (torch.tensor(v, dtype=torch.int32).cuda() for v in (lens, starts))
    got = ops.gemm.encoder_layers(x0.clone(), dl, ds, S, nh, d, 1e-12, layers)
    x, y = x0.clone(), x0.double().cpu()
    for L in layers:
        a = ops.encoder_attention(ops.gemm.linear_bias(x, L["wqkv"], L["bqkv"]), dl, len(lens), S, nh, d, starts=ds)
        x = ops.layer_norm(ops.gemm.linear_bias_residual(a, L["wo"], L["bo"], x), *L["ln1"], 1e-12)
        f = ops.gemm.linear_bias(x, L["w1"], L["b1"], gelu=True)
        x = ops.layer_norm(ops.gemm.linear_bias_residual(f, L["w2"], L["b2"], x), *L["ln2"], 1e-12)
        D = {k: tuple(t.double().cpu() for t in v) if isinstance(v, tuple) else v.double().cpu() for k, v in L.items()}
        q, k, v = F.linear(y, D["wqkv"], D["bqkv"]).view(T, 3, nh, d).unbind(1)
        a = torch.cat([F.scaled_dot_product_attention(*(t[s:s + n].transpose(0, 1) for t in (q, k, v))).transpose(0, 1).reshape(n, H)
                       for s, n in zip(starts, lens) if n])
        y = F.layer_norm(y + F.linear(a, D["wo"], D["bo"]), (H,), *D["ln1"], 1e-12)
        y = F.layer_norm(y + F.linear(F.gelu(F.linear(y, D["w1"], D["b1"])), D["w2"], D["b2"]), (H,), *D["ln2"], 1e-12)
    if len(lens) == 1:
        assert torch.equal(got, x)
    rms = lambda t: float((t.cpu().double() - y).square().mean().sqrt())  # noqa: E731
    assert rms(got) <= 1.1 * rms(x) + 1e-9, (rms(got), rms(x))


@pytest.mark.parametrize("lens,bad", [([9, 7], 0), ([9, 7], 1), ([1] * 16, 5), ([3, 1, 0, 4, 8], 3), ([16], 0), ([5, 0, 2], 2)])
@pytest.mark.parametrize("nh,d,inter", [(12, 32, 1536), (6, 64, 320), (3, 64, 128), (5, 32, 64)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_not_finite_rows_of_few_stay_in_their_text(lens, bad, nh, d, inter, value):
    """One row of one text is not finite: that text's rows are lost, every other text's are the bits they are without it."""
    torch.manual_seed(sum(lens) + inter)
    H, T, S = nh * d, sum(lens), max(lens)
    layers = [dict(wqkv=_b(3 * H, H, scale=0.05), bqkv=_b(3 * H), wo=_b(H, H, scale=0.05), bo=_b(H), ln1=(_b(H) + 1, _b(H)), w1=_b(inter, H, scale=0.05),
                   b1=_b(inter), w2=_b(H, inter, scale=0.05), b2=_b(H), ln2=(_b(H) + 1, _b(H))) for _ in range(2)]
    x, starts = _b(T, H), [sum(lens[:i]) for i in range(len(lens))]
    dl, ds = (torch.tensor(v, dtype=torch.int32).cuda() for v in (lens, starts))
    want = ops.gemm.encoder_layers(x.clone(), dl, ds, S, nh, d, 1e-12, layers)
    x[starts[bad] + lens[bad] - 1, 7] = value
    got = ops.gemm.encoder_layers(x.clone(), dl, ds, S, nh, d, 1e-12, layers)
    mine = torch.zeros(T, dtype=torch.bool, device="cuda")
    mine[starts[bad]:starts[bad] + lens[bad]] = True
    assert torch.isfinite(want).all() and got[mine].isnan().all() and torch.equal(got[~mine], want[~mine])
