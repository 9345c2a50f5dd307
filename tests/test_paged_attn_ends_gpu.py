"""Decode attention of 64-wide heads, where eight waves meet at once (csrc/kernels/attention.hip), against a double's: waves without keys, tiles of all head
groups, sequences whole and in parts, an output at an odd address."""
import numpy as np
import pytest
import torch

from distributed_llm_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,nkv", [(1, 1), (4, 2), (16, 4), (16, 2), (16, 1)])
@pytest.mark.parametrize("ctxs", [[1], [16, 17, 31, 32, 33], [255, 256, 257], [1000, 2, 511, 512, 513]])
def test_against_64_bits(nq, nkv, ctxs):
    torch.manual_seed(nq + len(ctxs))
    B, d, z = len(ctxs), 64, 16
    nb = -(-max(ctxs) // 16)
    kc, vc = torch.randn(B * nb, nkv, 16, d, device="cuda").bfloat16(), torch.randn(B * nb, nkv, d, 16, device="cuda").bfloat16()
    bt = torch.randperm(B * nb, device="cuda").view(B, nb).int()
    q = torch.randn(B, nq, d, device="cuda").bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    order = np.argsort(-np.array(ctxs), kind="stable")
    want, size = [], []
    for b, n in enumerate(ctxs):
        k = kc[bt[b].long()].permute(1, 0, 2, 3).reshape(nkv, -1, d)[:, :n].double().cpu().repeat_interleave(nq // nkv, 0)
        v = vc[bt[b].long()].permute(1, 0, 3, 2).reshape(nkv, -1, d)[:, :n].double().cpu().repeat_interleave(nq // nkv, 0)
        p = torch.softmax((q[b].double().cpu()[:, None] * k).sum(-1) * d ** -0.5, -1)[:, :, None]
        want.append((p * v).sum(1))
        size.append((p * v.abs()).sum(1))
    want, size = torch.stack(want), torch.stack(size)
    for chunk in (1024, 96):
        items = ops.decode_work_items(np.array(ctxs)[order], nkv, z, 1 << 20, min_chunk=chunk, seq=order, qstart=order)
        ws = (torch.empty(B * nkv * z * 16 * d, device="cuda"), torch.empty(B * nkv * z * 16 * 2, device="cuda"),
              torch.zeros(B * nkv + 2, dtype=torch.int32, device="cuda"))
        whole = torch.zeros(B * nq * d + 1, dtype=torch.bfloat16, device="cuda")
        for out in (None, whole[1:].view(B, nq, d)):
            kw = {} if out is None else {"out": out}
            got = ops.paged_attention(q, kc, vc, bt, i32(list(range(B))), i32([1] * B), i32(ctxs), i32(order.tolist()), i32([0] * B), splits=z,
                                      workspace=ws, items=torch.tensor(items, device="cuda"), grid_items=64, **kw)
            # weights rounded to 8 bits, then the result
            assert ((got.cpu().double().view(B, nq, d) - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -8 * size).all()
