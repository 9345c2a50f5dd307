"""Scratch of the chunk-parallel recurrences: bounded, heads or channels taken some at a time past the bound, with the same bits."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"
MB = 1 << 20


def i32(*v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def grown(f):
    """Result of f and the bytes it took beyond what it returns."""
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    at = torch.cuda.memory_allocated()
    y = f()
    torch.cuda.synchronize()
    return y, torch.cuda.max_memory_allocated() - at - y.numel() * y.element_size()


def test_retention():
    """24 heads of 128 x 128 over 16500 tokens: 260 chunks of 1.5 MB."""
    torch.manual_seed(0)
    T, H, d = 16500, 24, 128
    x = torch.randn(T, 4 * H * d, device=DEV).bfloat16()
    dec, pos, table = torch.linspace(0.9, 0.999, H, device=DEV), torch.arange(T, dtype=torch.int32, device=DEV), ops.rope_cos_sin(T, 64, 10000.0, DEV)
    m = (i32(0, 9000), i32(9000, T - 9000), i32(9000, T - 9000), i32(1, 0))
    st = torch.zeros(2, H, d, d, device=DEV)
    y, took = grown(lambda: seqmix.retention(x, H, d, d, table, 64, dec, st, 1e-6, pos, *m))
    assert took <= 257 * MB + T * H * d * 4          # the chunk states, and the outputs before their norm
    for h in (0, 12, 23):                            # a head by itself
        one = torch.cat([x.view(T, 4, H, d)[:, i, h] for i in range(4)], 1)
        s1 = torch.zeros(2, 1, d, d, device=DEV)
        z = seqmix.retention(one, 1, d, d, table, 64, dec[h:h + 1], s1, 1e-6, pos, *m)
        assert torch.equal(z, y[:, h * d:(h + 1) * d]) and torch.equal(s1[:, 0], st[:, h])


def test_scan():
    """4096 channels of 32 states over 20000 tokens: 626 chunks of 528 KB."""
    torch.manual_seed(1)
    T, C, N, R = 20000, 4096, 32, 8
    dt = torch.bfloat16
    xc, raw, dbc, xz = (torch.randn(T, w, device=DEV).to(dt) for w in (C, C, R + 2 * N, 2 * C))
    A, b, D = -torch.rand(C, N, device=DEV) * 4, torch.randn(C, device=DEV) - 3, torch.randn(C, device=DEV)
    m = (i32(0, 15000), i32(15000, T - 15000), i32(15000, T - 15000), i32(1, 0))
    st, cv = torch.zeros(2, C, N, device=DEV), torch.zeros(2, 3, C, device=DEV, dtype=dt)
    y, took = grown(lambda: seqmix.selective_scan(xc, raw, b, A, dbc, R, D, xz, st, cv, *m))
    assert took <= 257 * MB
    for c0 in (0, 1700, C - 256):                    # 256 channels by themselves
        c = slice(c0, c0 + 256)
        s1, v1 = torch.zeros(2, 256, N, device=DEV), torch.zeros(2, 3, 256, device=DEV, dtype=dt)
        z = seqmix.selective_scan(xc[:, c].contiguous(), raw[:, c].contiguous(), b[c], A[c], dbc, R, D[c],
                                  torch.cat([xz[:, c], xz[:, C + c0:C + c0 + 256]], 1), s1, v1, *m)
        assert torch.equal(z, y[:, c]) and torch.equal(s1, st[:, c]) and torch.equal(v1, cv[:, :, c])


def test_no_sequence():
    """Tokens of no sequence only: zeros, in chunks as token by token."""
    n = torch.zeros(0, dtype=torch.int32, device=DEV)
    H, dv, N = 2, 32, 16
    xbc, proj, v = torch.randn(130, H * dv + 2 * N, device=DEV), torch.randn(130, H, device=DEV), torch.ones(H, device=DEV)
    for chunked in (False, True):
        assert not seqmix.ssd_scan(xbc, proj, 0, H, dv, N, 1, v, -v, v, torch.zeros(1, H, N, dv, device=DEV), n, n, n, n, chunked=chunked).any()
