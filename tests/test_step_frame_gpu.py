"""The launches a decode step begins and ends with: its inputs and block-table updates, embedding rows, the sampler."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 5, 256, 257])
@pytest.mark.parametrize("V", [3, 8, 1000, 32000, 33003])
def test_greedy_rows(B, V):
    """Ties to the lowest index, -inf, NaN never chosen, rows of nothing else; the pinned copy; sampled rows between them."""
    g = torch.Generator().manual_seed(B + V)
    x = torch.randn(B, (V + 7) // 8 * 8, generator=g).mul_(4).round_().div_(4)[:, :V]      # many ties
    x[B // 2] = -float("inf")
    if B > 2:
        x[1, : V // 2] = float("nan")
        x[2] = float("nan")
        x[2, V - 1] = -float("inf")
    x = x.to(torch.bfloat16)
    buf = torch.zeros(B, (V + 7) // 8 * 8, dtype=torch.bfloat16, device="cuda")
    lg = buf[:, :V]
    lg.copy_(x)
    temp, one, k = torch.zeros(B, device="cuda"), torch.ones(B, device="cuda"), torch.ones(B, dtype=torch.int32, device="cuda")
    temp[3:4] = 1.0      # a sampled row of one candidate: its largest entry, whose index may be any of the tied ones
    seed, host = torch.tensor([7], dtype=torch.int32, device="cuda"), torch.full((B + 1,), -1, dtype=torch.int32).pin_memory()
    got = ops.sample_rows(lg, temp, one, k, seed, host=host).cpu()
    torch.cuda.synchronize()
    assert torch.equal(host[:B], got) and host[B] == -1
    for b in range(B):
        r = x[b].float()
        ok = r[~r.isnan()]
        want = int((r == ok.max()).nonzero()[0]) if ok.numel() else 0
        assert int(got[b]) == want if b != 3 else r[int(got[b])] == ok.max(), b


@pytest.mark.parametrize("shards", [2, 8])
def test_split_rows_pinned_copy(shards):
    x = torch.randn(3, 65536, device="cuda").to(torch.bfloat16)
    x[1, 5] = x[1, 60000] = 100.0
    z = lambda v, t=torch.float32: torch.full((3,), v, dtype=t, device="cuda")  # noqa: E731
    host, seed = torch.full((3,), -1, dtype=torch.int32).pin_memory(), torch.tensor([7], dtype=torch.int32, device="cuda")
    for temp in (0.0, 0.8):
        got = ops.sample_rows(x, z(temp), z(0.9), z(40, torch.int32), seed, shards=shards, host=host)
        assert torch.equal(got, ops.sample_rows(x, z(temp), z(0.9), z(40, torch.int32), seed, shards=1))
        assert torch.equal(host, got.cpu())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,scale,norm", [(1, 4, 1.0, True), (7, 1024, 1.0, True), (3, 1028, 12.5, True), (5, 5000, 1.0, False), (2, 8192, 0.5, True)])
def test_embed_rows(T, W, scale, norm, dtype):
    """Bit for bit the gather, widening and norm as launches of their own; an id outside the table is a row of zeros."""
    table = torch.randn(50, W, device="cuda").to(dtype)
    ids = torch.randint(0, 50, (T,), device="cuda", dtype=torch.int32)
    x, x2 = (torch.full((T, W), float("nan"), device="cuda") for _ in range(2))
    lp, h = (torch.full((T, W), float("nan"), device="cuda", dtype=dtype) for _ in range(2))
    w = torch.randn(W, device="cuda") if norm else None
    assert seqmix.embed_rows(ids, table, scale, x, x2, lp, w, 1e-6, h if norm else None)
    want = table[ids.long()].float() * scale
    assert torch.equal(x, want) and torch.equal(x2, want) and torch.equal(lp, want.to(dtype))
    if norm:
        hw = torch.empty_like(h)
        seqmix.scaled_resadd_rms(want, 1e-6, w=w, out=hw)
        assert torch.equal(h, hw)
    ids[-1] = 50
    assert seqmix.embed_rows(ids, table, scale, x)
    assert not x[-1].any()


def test_embed_rows_of_other_widths():
    """No vectors in a row: nothing is written, the caller's own launches run."""
    x = torch.full((1, 6), 3.0, device="cuda")
    assert not seqmix.embed_rows(torch.zeros(1, dtype=torch.int32, device="cuda"), torch.randn(4, 6, device="cuda"), 1.0, x)
    assert bool((x == 3.0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_embed_rows_of_any_ids(dtype):
    """Whole numbers of another width and strided ones, as the gather takes them; ids of other shapes go its way."""
    table, x = torch.randn(50, 64, device="cuda").to(dtype), torch.empty(6, 64, device="cuda")
    ids = torch.randint(0, 50, (6, 2), device="cuda")
    for some in (ids[:, 0], ids[:, 1].int(), ids[:, 0].to(torch.int16)):
        assert seqmix.embed_rows(some, table, 2.0, x.zero_())
        assert torch.equal(x, table[some.long()].float() * 2.0)
    assert not seqmix.embed_rows(ids[:, :1], table, 2.0, x)


@pytest.mark.parametrize("n", [0, 1, 64])
def test_updates_with_the_inputs(n):
    """The block-table pairs of the pinned buffer, as many as it says."""
    R, ids = 64, 8
    host = torch.zeros(2 * ids + 1 + 2 * R, dtype=torch.int32).pin_memory()
    off = 2 * ids
    host[ids:off] = -1
    at = torch.randperm(500)[:R].int()
    host[off] = n
    host[off + 1::2], host[off + 2::2] = at, torch.arange(R, dtype=torch.int32) + 1000
    dev, table, want = torch.zeros_like(host, device="cuda"), torch.zeros(500, dtype=torch.int32, device="cuda"), torch.zeros(500, dtype=torch.int32)
    ops.step_fetch(host, dev, 0, ids, ids, torch.zeros(ids + 1, dtype=torch.int32, device="cuda"), updates=(table, off, R))
    want[at[:n].long()] = torch.arange(n, dtype=torch.int32) + 1000
    assert torch.equal(table.cpu(), want) and torch.equal(dev.cpu(), host)
    with pytest.raises(RuntimeError):
        ops.step_fetch(host, dev, 0, ids, ids, torch.zeros(ids + 1, dtype=torch.int32, device="cuda"), updates=(table, off, R + 1))
