"""The GELU of values that end in bf16, in every kernel that has one, on every finite bf16 value: the bf16 number next to the exact one."""
import pytest
import torch

from distributed_llm_amd import ops
from distributed_llm_amd.ops import gemm as G

pytestmark = pytest.mark.gpu
SMALL, WIDE = (64, 64, 3, 1, 1, 4), (256, 256, 2, 1, 1, 4)


def values():
    v = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    return v[v.isfinite()]      # 65280


def projected(form):
    """x W^T with the values in W's first column and ones in x's."""
    v, K = values().cuda(), 64 if form != "decode" else 128
    w = torch.zeros(v.numel(), K, dtype=torch.bfloat16, device="cuda")
    w[:, 0] = v
    M = {"rows": 1, "few": 20}.get(form, 70 if form != "decode" else 5)
    x = torch.zeros(M, K, dtype=torch.bfloat16, device="cuda")
    x[:, 0] = 1
    bias = torch.zeros(v.numel(), dtype=torch.bfloat16, device="cuda")
    if form == "decode":
        y = torch.empty(M, v.numel(), dtype=torch.bfloat16, device="cuda")
        G.dgemm(x, G.frag_weight(w), v.numel(), G.DG_GELU, (1, 1, 1), y=y)
        return y
    if form in ("small", "wide"):
        y = torch.empty(M, v.numel(), dtype=torch.bfloat16, device="cuda")
        G._tgemm(ops._load(), x, w, G.EPI_GELU, SMALL if form == "small" else WIDE, y=y, bias=bias)
        return y
    return G.linear_bias(x, w, bias, gelu=True)


@pytest.mark.parametrize("form", ["elementwise", "gelu_erf", "gelu_erf ragged", "rows", "few", "small", "wide", "decode"])
def test_every_value(form):
    v = values()
    d = v.double()
    want = (0.5 * d * torch.special.erfc(-d * 0.5 ** 0.5)).to(torch.bfloat16).float()
    if form == "elementwise":
        got = ops.gelu(v.cuda()[None])
    elif form.startswith("gelu_erf"):
        from distributed_llm_amd.ops import seqmix
        got = seqmix.gelu_erf(v.cuda()[None] if " " not in form else torch.cat([v, v[:3]]).cuda()[None])[:, :v.numel()]
    else:
        got = projected(form)
    for row in got.float().cpu():
        # (numbers below the smallest normal f32 may be zero)
        bad = (row != want) & ~((want.abs() < 2.0 ** -125) & (row.abs() < 2.0 ** -125))
        assert not bad.any(), (v[bad][:5], row[bad][:5], want[bad][:5])


def test_what_is_not_finite():
    x = torch.tensor([[float("inf"), float("-inf"), float("nan"), 0.0, -0.0, 300.0, -300.0, 1.0]], device="cuda", dtype=torch.bfloat16)
    y = ops.gelu(x)[0].float().cpu()
    assert y[0] == float("inf") and y[1].isnan() and y[2].isnan() and y[3] == 0 and y[4] == 0 and y[5] == 300 and y[6] == 0
