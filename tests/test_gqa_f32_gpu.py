"""f32 attention over paged keys on the matrix cores, against 64 bits and against the general kernel (pages of 8 keys take it)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from distributed_llm_amd.models.llama import AttnMeta  # noqa: E402
from distributed_llm_amd.ops import ref, seqmix  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("H,G,GV,d,dv", [(16, 4, 4, 64, 64), (40, 2, 1, 128, 128), (3, 3, 3, 4, 5), (4, 2, 2, 68, 20), (2, 1, 1, 20, 100)])
@pytest.mark.parametrize("qlens,ctxs", [([1, 1, 1], [1, 16, 700]), ([1] * 40, [33] * 40), ([17, 0, 130], [17, 5, 145])])
@pytest.mark.parametrize("form", ["plain", "window", "kept", "chunk", "cap", "sinks", "slopes", "headgate"])
def test_f32_attention(H, G, GV, d, dv, qlens, ctxs, form):
    """One page up to many more than waves, rows without a key in a wave, one and several groups of 16 heads, widths that fill no
    block of 16, few and many workgroups; unwritten places of the last page hold NaN."""
    torch.manual_seed(5)
    S, T = len(qlens), sum(qlens)
    nb = [-(-c // 16) for c in ctxs]
    order = torch.randperm(sum(nb), device=DEV).to(torch.int32)
    bt, at = torch.zeros(S, max(nb), dtype=torch.int32, device=DEV), 0
    kc, vc = torch.randn(sum(nb), G, 16, d, device=DEV), torch.randn(sum(nb), GV, dv, 16, device=DEV)
    for s, (m, c) in enumerate(zip(nb, ctxs)):
        bt[s, :m] = order[at:at + m]
        at += m
        if c % 16:
            kc[bt[s, m - 1].long(), :, c % 16:] = float("nan")
            vc[bt[s, m - 1].long(), :, :, c % 16:] = float("nan")
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    qstart, qlen, ctx = i32([sum(qlens[:s]) for s in range(S)]), i32(qlens), i32(ctxs)
    q = torch.randn(T, H, d, device=DEV) * d ** -0.5
    gate = torch.randn(T, H if form == "headgate" else H * dv, device=DEV)
    kw = {"plain": {}, "window": {"window": 37}, "kept": {"window": 20, "keep_first": 5}, "chunk": {"chunk": 24}, "cap": {"softcap": 3.0},
          "sinks": {"sinks": torch.randn(H, device=DEV)}, "slopes": {"slopes": torch.rand(H, device=DEV)}, "headgate": {}}[form]
    clean = lambda x: torch.nan_to_num(x).double()  # noqa: E731
    w64 = {k: v.double() if torch.is_tensor(v) else v for k, v in kw.items()}
    want = ref.paged_gqa_attention(q.double(), clean(kc), clean(vc), bt, qstart, qlen, ctx, gate.double(), w64.get("window", 0), False,
                                   w64.get("keep_first", 0), 0.0, w64.get("chunk", 0), w64.get("softcap", 0.0), w64.get("sinks"),
                                   None, w64.get("slopes"))
    meta = AttnMeta(slots=None, block_tables=bt, qstart=qstart, qlen=qlen, ctx=ctx, tile_seq=None, tile_tok0=None, last_idx=None,
                    host_qlen=qlens)
    ts, tt = meta.latent_tiles(1, DEV, seqmix.gqa_tokens_per_tile(H, G, False))
    half = lambda x, keys: x.unflatten(keys, (2, 8)).movedim(keys, 1).flatten(0, 1).contiguous()  # noqa: E731
    errs = []
    for k, v, t in ((kc, vc, bt), (half(kc, 2), half(vc, 3), torch.stack((2 * bt, 2 * bt + 1), 2).flatten(1).contiguous())):
        got = seqmix.paged_gqa_attention(q, k, v, t, qstart, qlen, ctx, ts, tt, gate, **kw)
        assert torch.isfinite(got).all()
        errs.append(float((got.double() - want).norm() / want.norm()))
    # a score's rounding (d products) and an exponential's enter every weight: a few units of 2^-24; no worse than the general kernel's
    assert errs[0] < 2e-6 and errs[0] < 1.3 * errs[1] + 2.0 ** -24, errs


@pytest.mark.parametrize("n", [3, 70])      # eight waves share a workgroup's keys up to a round of the CUs, four past it
@pytest.mark.parametrize("H,G,d,dv", [(8, 8, 64, 64), (6, 2, 16, 3), (16, 4, 64, 128), (16, 1, 128, 33), (5, 5, 100, 64)])
def test_outputs_and_gates_of_a_tile(n, H, G, d, dv):
    """What a workgroup leaves at its end: every output of its rows once and nothing beside them, in tiles that are part full; gates by entry and by head
    out of wider rows, asked for ahead of the keys, are the sigmoid of their own entry."""
    torch.manual_seed(n)
    qlens = [1 + (5 * i) % 23 for i in range(n)]
    ctxs = [c + (7 * i) % 40 for i, c in enumerate(qlens)]
    T, nb = sum(qlens), [-(-c // 16) for c in ctxs]
    bt, at = torch.zeros(n, max(nb), dtype=torch.int32, device=DEV), 0
    for s, m in enumerate(nb):
        bt[s, :m] = torch.arange(at, at + m)
        at += m
    kc, vc, q = torch.randn(at, G, 16, d, device=DEV), torch.randn(at, G, dv, 16, device=DEV), torch.randn(T, H, d, device=DEV) * d ** -0.5
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    qs, ql, cx = i32([sum(qlens[:s]) for s in range(n)]), i32(qlens), i32(ctxs)
    meta = AttnMeta(slots=None, block_tables=bt, qstart=qs, qlen=ql, ctx=cx, tile_seq=None, tile_tok0=None, last_idx=None, host_qlen=qlens)
    a = (q, kc, vc, bt, qs, ql, cx, *meta.latent_tiles(1, DEV, seqmix.gqa_tokens_per_tile(H, G, False)))
    wide = torch.randn(T, H * dv + 7, device=DEV)
    plain = ref.paged_gqa_attention(q.double(), kc.double(), vc.double(), bt, qs, ql, cx)
    for gate in (None, wide[:, 3:H * dv + 3], wide[:, 2:H + 2]):
        odd = torch.full((T, H * dv + 6), 7.0, device=DEV)
        seqmix.paged_gqa_attention(*a, gate, out=odd[:, 5:H * dv + 5])
        want = plain if gate is None else plain * torch.sigmoid(gate.double() if gate.shape[1] == H * dv else gate.double().repeat_interleave(dv, 1))
        assert (odd[:, :5] == 7).all() and (odd[:, H * dv + 5:] == 7).all()
        # f32 sums of up to 62 keys and products of up to 128 dims, 2^-24 a term and in any direction; one more rounding for the gate
        assert (odd[:, 5:H * dv + 5].double() - want).abs().max() <= 2.0 ** -19
