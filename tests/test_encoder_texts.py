"""Texts to unit vectors in one call (embeddings in the first launch up to 16 rows, the mean in the last LayerNorm's) against one call per part."""
import pytest
import torch

from distributed_llm_amd import ops

pytestmark = pytest.mark.gpu


def _b(*s, scale=1.0):
    return (torch.randn(*s, device="cuda") * scale).to(torch.bfloat16)


@pytest.mark.parametrize("lens", [[1], [16], [9, 7], [1, 0, 12], [17], [0, 33, 31, 32, 1], [70, 30, 5, 64] * 8, [256, 100]])
@pytest.mark.parametrize("nh,d,inter", [(12, 32, 1536), (2, 32, 96), (3, 32, 256), (8, 64, 512), (10, 64, 640)])      # rows of up to 512 and past them
def test_against_the_parts(lens, nh, d, inter):
    torch.manual_seed(sum(lens) + inter)
    H, T, S, vocab = nh * d, sum(lens), max(lens), 100
    layers = [dict(wqkv=_b(3 * H, H, scale=0.05), bqkv=_b(3 * H), wo=_b(H, H, scale=0.05), bo=_b(H), ln1=(_b(H) + 1, _b(H)), w1=_b(inter, H, scale=0.05),
                   b1=_b(inter), w2=_b(H, inter, scale=0.05), b2=_b(H), ln2=(_b(H) + 1, _b(H))) for _ in range(2)]
    emb = (_b(vocab, H), _b(512, H), _b(H), _b(H) + 1, _b(H))
    ids = torch.randint(-3, vocab + 3, (T,), dtype=torch.int32).cuda()      # (ids outside the table are those at its ends)
    at = torch.tensor([p for n in lens for p in range(n)], dtype=torch.int32).cuda()
    starts = [sum(lens[:i]) for i in range(len(lens))]
    dl, ds = (torch.tensor(v, dtype=torch.int32).cuda() for v in (lens, starts))
    for bad in (False, True):
        if bad:
            ids[-1] = 7
            emb[0][7, 3] = float("nan")
        want = ops.embed_ln(ids, *emb, S, 1e-12, at)
        want = ops.mean_pool_l2(ops.gemm.encoder_layers(want, dl, ds, S, nh, d, 1e-12, layers), dl, ds)
        got = ops.gemm.encoder_texts(ids, at, emb, dl, ds, S, nh, d, 1e-12, layers)
        assert torch.equal(got.isnan(), want.isnan()) and bool(got.isnan().any()) == bad
        # equal rows; n of them summed in f32 in another order: unit vectors n 2^-24 apart at most
        torch.testing.assert_close(got, want, rtol=0, atol=max(lens) * 2.0 ** -24, equal_nan=True)
        assert all(not got[i].any() for i, n in enumerate(lens) if n == 0)
