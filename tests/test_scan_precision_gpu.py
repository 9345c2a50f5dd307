"""SiLU and softplus inside the recurrences' kernels: as exact in the forms for prompts and steps as in the general ones, whose formulas are
x / (1 + e^-x) and log(1 + e^x) in f32."""
import pytest
import torch

from distributed_llm_amd.ops import seqmix

pytestmark = pytest.mark.gpu
DEV = "cuda"
RANGES = [(-60.0, -20.0), (-20.0, -5.0), (-5.0, -1.0), (-1.0, -1e-3), (1e-3, 1.0), (1.0, 5.0), (5.0, 20.0), (20.0, 60.0)]


def error(got, want):
    """Root mean square of the relative error in units of 2^-24."""
    return float(((got.double() - want) / want).pow(2).mean().sqrt()) * 2 ** 24


def one_token_each(S):
    n = torch.arange(S, dtype=torch.int32, device=DEV)
    one = torch.ones_like(n)
    return n, one, one, n


@pytest.mark.parametrize("lo,hi", RANGES)
def test_scan(lo, hi):
    """A = 0, B = x = 1: a state is its step size.  B = 0, D = x = 1: an output is SiLU of its gate."""
    torch.manual_seed(1)
    S, C = 64, 4096
    x = torch.rand(S, C, device=DEV) * (hi - lo) + lo
    ones, z = torch.ones(S, C, device=DEV), torch.zeros(C, device=DEV)
    step, gate = torch.nn.functional.softplus(x.double(), threshold=1e9), x.double() * torch.sigmoid(x.double())
    step = torch.where(x < 0, torch.log1p(torch.exp(x.double())), step)
    errs = {}
    for name, N, chunked in (("general", 2, False), ("step", 4, False), ("prompt", 4, True)):
        conv = torch.zeros(S, 3, C, device=DEV)
        A, st = torch.zeros(C, N, device=DEV), torch.zeros(S, C, N, device=DEV)
        seqmix.selective_scan(ones, x, z, A, torch.ones(S, 2 * N, device=DEV), 0, z, torch.ones(S, 2 * C, device=DEV), st, conv,
                              *one_token_each(S), chunked=chunked)
        y = seqmix.selective_scan(ones, x, z, A, torch.zeros(S, 2 * N, device=DEV), 0, z + 1, torch.cat([ones, x], 1), torch.zeros_like(st),
                                  conv, *one_token_each(S), chunked=chunked)
        errs[name] = error(st[:, :, 0], step), error(y, gate)
    for name in ("step", "prompt"):
        for e, g in zip(errs[name], errs["general"]):
            assert e <= 1.02 * g + 1e-3, errs          # 262144 points: the figures repeat to a part in a thousand


@pytest.mark.parametrize("lo,hi", RANGES)
def test_lightning(lo, hi):
    """One token: the state is SiLU(k) SiLU(v), and SiLU(100) is 100."""
    torch.manual_seed(2)
    S, H, dv = 256, 8, 128
    v = torch.rand(S, H * dv, device=DEV) * (hi - lo) + lo
    qk = torch.full((S, 2 * H), 100.0, device=DEV)
    st = [torch.zeros(S, H, 1, dv, device=DEV) for _ in range(2)]
    for s, chunked in zip(st, (False, True)):
        seqmix.lightning_attention(torch.cat([qk, v, v], 1), H, 1, dv, torch.full((H,), 0.9, device=DEV), s, 1e-6, torch.ones(H * dv, device=DEV),
                                   *one_token_each(S), chunked=chunked)
    assert torch.equal(st[0], st[1])                   # prompts and steps of one layer round alike


@pytest.mark.parametrize("decay,more", [("slow", 0), ("model", 0), ("steep", 2)])
@pytest.mark.parametrize("H,G,d,dv", [(16, 8, 128, 128), (4, 2, 64, 64)])
def test_delta_tiles(decay, more, H, G, d, dv):
    """Sixteen tokens at a time against token by token: no further from 64 bits with decays near 1 or a model's (A of 1 to 16, steps
    of 0.001 to 0.1).  Where a token keeps a fiftieth of the state and a few roundings are all there is, two more (2^-24 / sqrt 3 root
    mean square each): a token's update times its decay up to the tile's end, and the sum over the tile."""
    torch.manual_seed(3)
    T = 385
    qkv, gba = torch.randn(T, 2 * G * d + H * dv, device=DEV), torch.randn(T, H * dv + 2 * H, device=DEV)
    na, dtb, nw = -torch.rand(H, device=DEV) * {"slow": 0.05, "model": 0.0, "steep": 8.0}[decay], torch.randn(H, device=DEV), torch.randn(dv, device=DEV)
    if decay == "model":
        step = torch.exp(torch.rand(H, device=DEV) * 4.6 - 6.9)
        na, dtb = -(1 + 15 * torch.rand(H, device=DEV)), step + torch.log(-torch.expm1(-step))
    q, k, v = qkv.double().split([G * d, G * d, H * dv], 1)
    q, k = (z.view(T, G, d) * torch.rsqrt((z.view(T, G, d) ** 2).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
    q, k = (q * d ** -0.5).repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
    v, gate, beta, al = v.view(T, H, dv), *gba.double().split([H * dv, H, H], 1)
    beta, g = torch.sigmoid(beta), torch.exp(na.double() * torch.nn.functional.softplus(al + dtb.double(), threshold=40))
    M, o = torch.zeros(H, dv, d, dtype=torch.float64, device=DEV), []
    for t in range(T):
        M = g[t, :, None, None] * M
        u = beta[t, :, None] * (v[t] - (M * k[t, :, None]).sum(-1))
        M = M + u[:, :, None] * k[t, :, None]
        o.append((M * q[t, :, None]).sum(-1))
    o = torch.stack(o)
    want = (o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6) * nw.double()).reshape(T, -1) * torch.nn.functional.silu(gate)
    i32 = lambda x: torch.tensor([x], dtype=torch.int32, device=DEV)  # noqa: E731
    errs = []
    for tiled in (True, False):
        st = torch.zeros(1, H, dv, d, device=DEV)
        y = seqmix.delta_rule(qkv, gba, H, G, d, dv, na, dtb, nw, 1e-6, st, i32(0), i32(T), i32(T), i32(0), tiled=tiled)
        errs.append((float((y.double() - want).norm() / want.norm()), float((st[0].double() - M).norm() / M.norm())))
    assert all(a * a <= b * b + more * 2.0 ** -48 / 3 for a, b in zip(*errs)), errs
