"""The tiled GEMM's QKV epilogue over prompts: runs of eight consecutive cache slots (written as vectors) among rows that are alone,
runs cut by a tile's edge, by another sequence or by rows without a slot."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.models.llama import fuse_qkv_weight
from distributed_llm_amd.ops import gemm as G
from distributed_llm_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"
PLANS = [(64, 64, 3, 1, 1, 4), (64, 64, 3, 1, 2, 4, 1, 0, 0, 64, 32), (64, 64, 3, 2, 1, 4), (128, 128, 3, 1, 1, 8), (192, 128, 3, 1, 1, 8),
         (256, 128, 3, 1, 1, 8, 1, 8, 0, 64, 16, 2), (256, 256, 2, 1, 1, 8, 1, 0, 0, 64, 16, 8), (256, 256, 4, 1, 1, 8, 1, 0, 0, 32),
         (256, 256, 2, 1, 1, 4), (256, 256, 2, 1, 1, 4, 1, 0, 0, 64, 16, 8)]


def _slots(kind, M):
    if kind == "prompt":        # three sequences behind each other, in blocks anywhere, the second from a position inside a block
        out, block = [], iter(torch.randperm(M // 8 + 8).tolist())
        for n, at in ((M // 3, 0), (M // 4, 5), (M - M // 3 - M // 4, 0)):
            b = None
            for p in range(at, at + n):
                b = next(block) if b is None or p % 16 == 0 else b
                out.append(16 * b + p % 16)
        return torch.tensor(out, dtype=torch.int32)
    s = torch.arange(M, dtype=torch.int32)
    if kind == "holes":
        s[3::11] = -1
    return s


@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("kind", ["prompt", "all", "holes"])
@pytest.mark.parametrize("M,d,nq,nkv", [(67, 64, 4, 2), (300, 32, 2, 1), (520, 128, 2, 2)])
def test_slots(plan, kind, M, d, nq, nkv):
    torch.manual_seed(M + d)
    G.reserve(DEV)
    H, N = 256, (nq + 2 * nkv) * d
    r, ln = torch.randn(M, H, device=DEV).bfloat16(), (1.0 + 0.1 * torch.randn(H, device=DEV)).bfloat16()
    wqkv = (torch.randn(N, H, device=DEV) * 0.05).bfloat16()
    wf, slots = fuse_qkv_weight(wqkv, ln, nq, nkv, d), _slots(kind, M)
    pos = torch.randint(0, 4000, (M,), dtype=torch.int32)
    cs, nblk = ops.rope_cos_sin(4096, d, 10000.0, DEV), int(slots.max()) // 16 + 1
    ssq = (r.float() ** 2).sum(1)[None].contiguous()
    kc, vc = torch.zeros(nblk, nkv, 16, d, device=DEV).bfloat16(), torch.zeros(nblk, nkv, d, 16, device=DEV).bfloat16()
    q = torch.empty(M, nq, d, device=DEV, dtype=torch.bfloat16)
    G._tgemm(G._native(r), r, wf, G.EPI_QKV, plan, ssq_in=ssq, ssq_n=1, norm_scale=1.0 / H, eps=1e-5, pos=pos.to(DEV), cos_sin=cs,
             slots=slots.to(DEV), q_out=q, kc=kc, vc=vc, nq=nq, nkv=nkv, d=d)
    qkv = (ref.rms_norm(r.cpu(), ln.cpu(), 1e-5).float() @ wqkv.cpu().float().t()).bfloat16()
    kr, vr = torch.zeros(nblk, nkv, 16, d).bfloat16(), torch.zeros(nblk, nkv, d, 16).bfloat16()
    qr = ref.rope_and_cache(qkv, pos, cs.cpu(), slots, kr, vr, nq, nkv, d)
    # the norm weight folded into bf16 columns and a rounding ahead of the rotation: 2^-7 of the largest value
    tol = 2.0 ** -7 * 2 * qkv.float().abs().max().item()
    for got, want in ((q, qr), (kc, kr), (vc, vr)):
        torch.testing.assert_close(got.cpu().float(), want.float(), atol=tol, rtol=2e-2)
        assert torch.equal(got.cpu() == 0, want == 0)      # nothing outside the slots
