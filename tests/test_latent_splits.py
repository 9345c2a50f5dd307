"""Key splits of latent attention: how many, and that a split more or less, or one without keys, changes a row by no more than its rounding."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import reference as ref
from distributed_llm_amd.ops import seqmix


def test_one_round_of_workgroups():
    for n in range(1, 600):
        sp = seqmix.latent_splits(n, 16)
        assert 1 <= sp <= 64 and (sp == 1 or n * sp <= 512) and (n > 128 or sp == min(64, 256 // n))
    assert [seqmix.latent_splits(n, 16) for n in (1, 4, 24, 128, 129, 170, 171, 400)] == [64, 64, 10, 2, 3, 3, 1, 1]
    assert seqmix.latent_splits(4, 8) == 64 and seqmix.latent_splits(40, 128) == 1      # (eight 16-row blocks an entry)


def test_rounds_of_the_device_and_of_the_vector_form():
    assert [seqmix.latent_splits(n, 16, cus=64) for n in (1, 4, 24, 32, 33, 42, 43, 100)] == [64, 16, 2, 2, 3, 3, 1, 1]
    assert [seqmix.latent_splits(n, 16, vector=1) for n in (1, 4, 5, 24, 48, 75, 100, 128, 150, 200, 219, 220, 256, 257, 900)] == \
        [64, 64, 51, 10, 5, 3, 5, 2, 3, 1, 1, 1, 1, 1, 1]
    assert [seqmix.latent_splits(n, 16, vector=2) for n in (1, 8, 9, 48, 150, 200, 256, 257, 400, 900)] == [64, 64, 56, 10, 3, 5, 2, 1, 1, 1]
    assert [seqmix.latent_vector_wgs(*r) for r in ((128, 32), (240, 0), (241, 0), (256, 32))] == [2, 2, 1, 1]


@pytest.mark.gpu
@pytest.mark.parametrize("H,rank,rd", [(16, 256, 32), (4, 128, 6), (32, 512, 64)])
def test_f32_splits_against_64_bits(H, rank, rd):
    """The vector form, whose tiles are 64 keys, or 32 at rank 512: splits with and without keys, more of them than tiles, the rule's own."""
    torch.manual_seed(H)
    dim, dev, ctxs = 32, "cuda", [1, 31, 64, 65, 700, 1025, 2300]
    n, per = len(ctxs), [(c + 15) // 16 for c in ctxs]
    I = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    bt, at = torch.zeros(n, max(per), dtype=torch.int32), 1
    for i, m in enumerate(per):
        bt[i, :m] = torch.arange(at, at + m)
        at += m
    cache = torch.randn(at, 16, rank + rd, device=dev)
    qa, q = torch.randn(H, n, rank, device=dev), torch.randn(n, H * (dim + rd), device=dev)
    table, pos, scale, sinks = ops.rope_cos_sin(4096, rd, 10000.0, torch.device(dev)), I([c - 1 for c in ctxs]), 0.05, torch.randn(H, device=dev)
    args = (qa, q, dim, rd, pos, table, cache, bt.to(dev), I(list(range(n))), I([1] * n), I(ctxs), I(list(range(n))), I([0] * n), scale)
    want = torch.empty(H, n, rank, dtype=torch.float64, device=dev)
    for i, c in enumerate(ctxs):
        kv = cache[bt[i, :per[i]].long().to(dev)].flatten(0, 1)[:c].double()
        cs, sn = (x.double() for x in ref._rot_table(table, pos[i:i + 1], rd // 2))
        qr = ref._rope_interleaved(q[i:i + 1].double().view(1, H, dim + rd)[..., dim:], cs[:, None], sn[:, None])[0]
        sc = torch.cat([(qa[:, i].double() @ kv[:, :rank].t() + qr @ kv[:, rank:].t()) * scale, sinks.double()[:, None]], 1)
        want[:, i] = torch.softmax(sc, 1)[:, :c] @ kv[:, :rank]
    one = None
    for splits in (1, 2, 10, 16, 33, 64, None):
        got = seqmix.latent_attention(*args, splits=splits, sinks=sinks)
        err = float((got - want).norm() / want.norm())
        one = err if one is None else one
        print("H %d rank %d splits %s: off by %.2g" % (H, rank, splits, err))
        assert err <= 4e-6 and err <= 1.5 * one      # f32 sums, whose shorter parts are no worse


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 2, 16, 17, 33, 64])
@pytest.mark.parametrize("sink", [False, True])
def test_splits_with_and_without_keys(splits, sink):
    torch.manual_seed(splits)
    H, dim, rd, rank, vd, ctxs = 16, 64, 32, 256, 64, [1, 64, 65, 700, 1025, 2300]
    n, dev = len(ctxs), "cuda"
    I = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    per = [(c + 15) // 16 for c in ctxs]
    bt = torch.zeros(n, max(per), dtype=torch.int32)
    at = 1
    for i, m in enumerate(per):
        bt[i, :m] = torch.arange(at, at + m)
        at += m
    cache = torch.randn(at, 16, rank + rd, device=dev).bfloat16()
    qa, q = torch.randn(H, n, rank, device=dev).bfloat16(), torch.randn(n, H * (dim + rd), device=dev).bfloat16()
    sinks = torch.randn(H, device=dev) if sink else None
    table = ops.rope_cos_sin(4096, rd, 10000.0, torch.device(dev))
    pos = I([c - 1 for c in ctxs])
    args = (qa, q, dim, rd, pos, table, cache, bt.to(dev), I(list(range(n))), I([1] * n), I(ctxs))
    got = seqmix.latent_attention(*args, I(list(range(n))), I([0] * n), 0.05, splits=splits, sinks=sinks)
    want = ref.latent_attention(*args, 0.05, False, sinks)
    # weights in two bf16 parts (2^-17), f32 sums, one rounding to 8 bits of values of about one
    torch.testing.assert_close(got.float(), want.float(), atol=2.0 ** -7, rtol=2.0 ** -7)
    uv = torch.randn(H, rank, vd, device=dev).bfloat16()
    if splits > 1:
        out = torch.empty(n, H * vd, device=dev, dtype=torch.bfloat16)
        seqmix.latent_attention(*args, I(list(range(n))), I([0] * n), 0.05, splits=splits, sinks=sinks, up=(uv, None, out))
        lat = torch.bmm(got.float(), uv.float()).transpose(0, 1).reshape(n, -1)
        torch.testing.assert_close(out.float(), lat, atol=2.0 ** -6 * rank ** 0.5, rtol=2.0 ** -7)
