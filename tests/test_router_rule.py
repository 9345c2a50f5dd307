"""Routers whose weights one workgroup reads fast enough take one launch, wider ones two, many rows of those the library's product."""
import types

import pytest
import torch

from distributed_llm_amd.ops import seqmix


@pytest.mark.parametrize("T,H,n,way", [(1, 1024, 8, "one"), (16, 2048, 64, "one"), (16, 8192, 8, "one"), (4096, 64, 8, "one"), (4097, 64, 8, "two"),
                                       (1, 1024, 65, "two"), (1, 4096, 64, "two"), (16, 1024, 256, "two"), (2, 8192, 256, "two"), (33, 1024, 256, "library"),
                                       (512, 8192, 64, "library"), (1, 64, 257, "library"), (0, 64, 8, "one")])
def test_router_rule(monkeypatch, T, H, n, way):
    took = []
    monkeypatch.setattr(seqmix, "_native", lambda x: types.SimpleNamespace(router_topk=lambda *a: took.append("two" if a[-1] else "one")))
    monkeypatch.setattr(seqmix, "route_topk", lambda *a: took.append("library") or (None, None, None))
    seqmix.router_topk(torch.zeros(T, H, dtype=torch.bfloat16), torch.zeros(n, H), n, 2)
    assert took == [way]


@pytest.mark.gpu
@pytest.mark.parametrize("T,H,n", [(1, 1024, 64), (5, 1032, 8), (16, 64, 33), (3, 4096, 32)])
def test_two_launches_same_bits(T, H, n):
    torch.manual_seed(H)
    x, w = torch.randn(T, H, device="cuda").bfloat16(), torch.randn(n, H, device="cuda") / H ** 0.5
    got = []
    for apart in (False, True):
        ids, wts, idw, lg = (torch.empty(T, m, device="cuda", dtype=d) for m, d in ((2, torch.int32), (2, torch.float32), (1, torch.float32), (n, torch.float32)))
        seqmix._native(x).router_topk(x, w, n, 2, 1, 1, 0, 0, None, n, ids, wts, idw.view(-1), lg, apart)
        got.append((ids, wts, idw, lg))
    assert all(torch.equal(a, b) for a, b in zip(*got))
