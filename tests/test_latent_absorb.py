"""The absorbed key up-projection of few tokens (latent.hip) against a double's, at the edges of its tiles; elsewhere the vendor's batched product."""
import pytest
import torch

from distributed_llm_amd.ops import seqmix


def test_on_the_cpu():
    q, uk = torch.randn(3, 2, 32), torch.randn(2, 32, 16)
    assert torch.equal(seqmix.latent_absorb(q, uk, uk.transpose(1, 2).contiguous()), torch.bmm(q.transpose(0, 1), uk))


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 64, 65])
@pytest.mark.parametrize("H,dim,rot,rank", [(1, 32, 0, 16), (16, 64, 32, 256), (3, 96, 8, 80), (5, 160, 0, 512), (2, 48, 16, 64), (2, 64, 4, 64), (2, 64, 0, 72)])
def test_against_64_bits(T, H, dim, rot, rank, monkeypatch):
    torch.manual_seed(T + rank)
    q = torch.randn(T, H * (dim + rot), device="cuda").bfloat16().view(T, H, dim + rot)[:, :, :dim]
    uk = (torch.randn(H, dim, rank, device="cuda") * dim ** -0.5).bfloat16()
    ran, ext = [], seqmix._native(q)
    monkeypatch.setattr(seqmix, "_native", lambda x: ran.append(1) or ext)
    got = seqmix.latent_absorb(q, uk, uk.transpose(1, 2).contiguous())
    assert bool(ran) == (T <= 64 and dim % 32 == 0 and rot % 8 == 0 and rank % 16 == 0)
    a, b = q.double().transpose(0, 1).contiguous(), uk.double()
    want, size = torch.bmm(a, b), torch.bmm(a.abs(), b.abs())
    # dim products summed in f32, one rounding to 8 bits
    assert got.shape == want.shape and ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + dim * 2.0 ** -23 * size).all()
