"""An infinity or NaN in one token of a prompt leaves the tokens before it, and the other sequences, as they are: the forms of the
recurrences that take 64 or 16 tokens at once multiply what a token does not see by zero, and zero times either is NaN.  The tokens
after it are lost in any form.  What is compared differs by the order of the sums only: 4e-6 relative as in the chunks' own tests."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix
from test_seqmix_gpu import batch

pytestmark = pytest.mark.gpu
DEV = "cuda"
QLENS, STARTS, BAD = [100, 45], [3, 0], 37


@pytest.fixture(autouse=True, scope="module")
def _native():
    assert ops.native_available(), "HIP extension must be built for GPU tests"


def same_before(run, x, cols, value):
    clean = run(x.clone()).double()
    x[BAD, cols] = value
    got = run(x).double()
    keep = [t for t in range(sum(QLENS)) if t < BAD or t >= QLENS[0]]
    assert torch.isfinite(got[keep]).all() and not torch.isfinite(got[BAD]).all()
    assert float((got[keep] - clean[keep]).norm() / clean[keep].norm()) < 4e-6


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["q", "k", "v"])
@pytest.mark.parametrize("act", [False, True])
def test_chunks(act, where, value):
    torch.manual_seed(71)
    H, d, dv = 2, 64, 128
    T, qstart, qlen, ctx, rows, pos = batch(QLENS, STARTS)
    x = torch.randn(T, 2 * H * d + 2 * H * dv, device=DEV)
    dec, st = torch.tensor([0.9, 0.99], device=DEV), torch.randn(2, H, d, dv, device=DEV)
    table, nw = ops.rope_cos_sin(512, d, 10000.0, DEV), torch.randn(H * dv, device=DEV)

    def run(x):
        if act:
            return seqmix.lightning_attention(x, H, d, dv, dec, st.clone(), 1e-5, nw, qstart, qlen, ctx, rows, chunked=True)
        return seqmix.retention(x, H, d, dv, table, d, dec, st.clone(), 1e-6, pos, qstart, qlen, ctx, rows, chunked=True)
    same_before(run, x, {"q": 5, "k": H * d + 5, "v": 2 * H * d + 21}[where], value)


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("where", ["q", "k", "v", "beta", "decay"])
def test_tiles(where, value):
    torch.manual_seed(72)
    H, G, d, dv = 2, 2, 128, 128
    T, qstart, qlen, ctx, rows, _ = batch(QLENS, STARTS)
    n = G * d
    x = torch.randn(T, 2 * n + H * dv + H * dv + 2 * H, device=DEV)
    split = 2 * n + H * dv
    na, dtb, nw = torch.tensor([-0.1, -0.3], device=DEV), torch.zeros(H, device=DEV), torch.ones(dv, device=DEV)
    st = torch.randn(2, H, dv, d, device=DEV)

    def run(x):
        return seqmix.delta_rule(x[:, :split].contiguous(), x[:, split:].contiguous(), H, G, d, dv, na, dtb, nw, 1e-6, st.clone(), qstart, qlen,
                                 ctx, rows, tiled=True)
    gba = split + H * dv
    if where in ("beta", "decay"):
        value = float("nan")      # infinite logits are a gate of 0 or 1
    same_before(run, x, {"q": 5, "k": n + 5, "v": 2 * n + 21, "beta": gba, "decay": gba + H}[where], value)
