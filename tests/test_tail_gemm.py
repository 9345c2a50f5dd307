"""A sublayer's tail in the launch of the product behind it (csrc/kernels/tail_gemm.hip) against the two launches it replaces: the stream and the
normed rows have their bits, and where K splits alike the product has too."""
import os
import re

import pytest
import torch

from distributed_llm_amd.ops import gemm as G
from distributed_llm_amd.ops import seqmix

from test_kernel_resources import HIPCC, _usage

GPU = pytest.mark.gpu
DEV = "cuda"


def rnd(*s, scale=1.0):
    return torch.randn(*s, device=DEV) * scale


def parts(M, N, K, glu, bias):
    torch.manual_seed(M * 1000 + N)
    y = rnd(M, K + 8).bfloat16()[:, :K]
    w = rnd(N, K, scale=K ** -0.5).bfloat16()
    return y, rnd(M, K), rnd(K), rnd(K), rnd(K) if bias else None, w, G.frag_weight(w, "glu" if glu else False)


@GPU
@pytest.mark.parametrize("M", [1, 3, 15, 16])
@pytest.mark.parametrize("N,K", [(16, 32), (72, 96), (1088, 1024), (4096, 512), (4104, 1024), (8192, 1024), (40, 992)])
@pytest.mark.parametrize("bias", [False, True])
def test_plain(M, N, K, bias):
    y, x, wp, wn, b, w, wf = parts(M, N, K, False, bias)
    assert G.tail_takes(y, w, wp, wn, b) and not G.tail_takes(y, torch.empty(32 * 256 + 16, K, device=DEV), wp)
    x2 = torch.full_like(x, float("nan"))
    out = G.Tail(y, wp, 1e-5, x, x2, wn, b).linear(w, wf)
    x1, h = x.clone(), torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    seqmix.resadd_norm(y, wp, 1e-5, x1, wn, h, bias=b)
    assert torch.equal(x2, x1)
    want = h.double() @ w.double().t()
    # f32 sums of K products, one rounding to 8 bits
    assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + K * 2.0 ** -22 * (h.abs().double() @ w.abs().double().t())).all()
    if K % 512 == 0:
        two = torch.empty_like(out)
        G.dgemm(h, wf, N, G.EPI_PLAIN, (1, 4, 4), y=two)
        assert torch.equal(out, two)


@GPU
@pytest.mark.parametrize("M", [1, 4, 16])
@pytest.mark.parametrize("N,K", [(16, 64), (5632, 1024), (4112, 512)])
@pytest.mark.parametrize("act,limit,alpha", [("clamped", 2.0, 1.702), ("gelu_tanh", 0.0, 1.0), ("swiglu", 0.0, 1.0)])
def test_gated(M, N, K, act, limit, alpha):
    y, x, wp, wn, b, w, wf = parts(M, N, K, True, True)
    ab = rnd(N)
    x2 = torch.empty_like(x)
    out = G.Tail(y, wp, 1e-5, x, x2, wn, b).linear(w, wf, act, ab, limit, alpha)
    x1, h = x.clone(), torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    seqmix.resadd_norm(y, wp, 1e-5, x1, wn, h, bias=b)
    two = torch.empty_like(out)
    G.dgemm(h, wf, N, G.DG_GLU, (1, 4, 4), y=two, bias=ab, mode=seqmix.GLU_MODES[act], limit=limit, alpha=alpha)
    assert torch.equal(x2, x1)
    if K % 512 == 0:
        assert torch.equal(out, two)
    else:      # another order of f32 sums: a rounding apart, ahead of the activation and behind it
        torch.testing.assert_close(out.float(), two.float(), atol=2.0 ** -6, rtol=2.0 ** -6)


@GPU
@pytest.mark.parametrize("K", [1056, 1024])
def test_not_taken(K):
    y, w = rnd(17 if K == 1024 else 4, K).bfloat16(), rnd(64, K).bfloat16()
    assert not G.tail_takes(y, w)
    assert not G.tail_takes(rnd(4, 64).bfloat16(), rnd(64, 64).bfloat16(), rnd(65)[1:])      # (a vector 4 bytes off)


@pytest.mark.parametrize("taps", [0, 3])
def test_an_input_convolution_reads_rows(monkeypatch, taps):
    """What a mixer's product takes along exists nowhere else: not where a convolution stands ahead of the mixer.  A feed-forward has none."""
    from types import SimpleNamespace as NS

    from distributed_llm_amd.models.hybrid import HybridModel
    monkeypatch.setattr(G, "tail_takes", lambda *a: True)
    monkeypatch.setattr(seqmix, "resadd_norm", lambda *a, **k: None)
    m = object.__new__(HybridModel)
    m.tap, m.dtype, m.cfg = None, torch.bfloat16, NS(rms_eps=1e-5, input_conv=taps)
    w, v, x = torch.zeros(64, 64, dtype=torch.bfloat16), torch.zeros(64), torch.zeros(2, 64)
    L = {"proj": w, "proj_r": w, "up": w, "up_act_r": w, "order_kept": False}
    taken = lambda S: isinstance(m._tail(w[:2], v, x, v, None, L, S)[1], G.Tail)  # noqa: E731
    assert taken(NS(mixer=NS(kind="mlstm"))) == (taps == 0) and taken(None)


@pytest.mark.parametrize("M,K,one", [(1, 64, True), (12, 512, True), (13, 512, False), (16, 256, False), (13, 576, True), (16, 1024, True)])
def test_rows_and_widths_of_one_launch(monkeypatch, M, K, one):
    from types import SimpleNamespace as NS

    from distributed_llm_amd.models.hybrid import HybridModel
    monkeypatch.setattr(G, "tail_takes", lambda *a: True)
    monkeypatch.setattr(seqmix, "resadd_norm", lambda *a, **k: None)
    m = object.__new__(HybridModel)
    m.tap, m.dtype, m.cfg = None, torch.bfloat16, NS(rms_eps=1e-5, input_conv=0)
    w, v = torch.zeros(64, K, dtype=torch.bfloat16), torch.zeros(K)
    L = {"up": w, "up_act_r": w, "order_kept": False}
    assert isinstance(m._tail(w[:M], v, torch.zeros(M, K), v, None, L)[1], G.Tail) == one


@GPU
def test_replays():
    """In a captured graph, with eager work between: the stream goes on from buffer to buffer."""
    y, x, wp, wn, b, w, wf = parts(4, 1024, 1024, False, True)
    xs, x0 = torch.empty(4, 1024, device=DEV), x.clone()

    def step():
        xs.copy_(x0)
        x2, x3 = torch.empty_like(xs), torch.empty_like(xs)
        o = G.Tail(y, wp, 1e-5, xs, x2, wn, b).linear(w, wf)
        return G.Tail(o, wp, 1e-5, x2, x3, wn, b).linear(w, wf), x3
    want = [t.clone() for t in step()]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = step()
    for _ in range(4):
        g.replay()
        rnd(1000).sum()
        torch.cuda.synchronize()
        assert all(torch.equal(a, c) for a, c in zip(got, want))


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_registers():
    out = _usage("tail_gemm.hip")
    assert "ScratchSize" in out and set(re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", out)) == {"0"}
