"""Prompt attention with a row to a lane column (gqa.hip: bf16 output, a value head to a key head) against 64 bits, and against the form with four rows a
lane, which f32 outputs still take: widths that fill no block, rows of one and several tokens, ragged tiles, kept keys, splits, outputs and gates that are
no whole vectors."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from distributed_llm_amd.models.llama import AttnMeta  # noqa: E402
from distributed_llm_amd.ops import ref, seqmix  # noqa: E402

DEV = "cuda"


def setup(H, G, d, dv, qlens, ctxs, seed=3):
    torch.manual_seed(seed)
    S, T, nb = len(qlens), sum(qlens), [-(-c // 16) for c in ctxs]
    order, at = torch.randperm(sum(nb), device=DEV).to(torch.int32), 0
    bt = torch.zeros(S, max(nb), dtype=torch.int32, device=DEV)
    for s, m in enumerate(nb):
        bt[s, :m] = order[at:at + m]
        at += m
    kc, vc = torch.randn(sum(nb), G, 16, d, device=DEV).bfloat16(), torch.randn(sum(nb), G, dv, 16, device=DEV).bfloat16()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    qs, ql, cx = i32([sum(qlens[:s]) for s in range(S)]), i32(qlens), i32(ctxs)
    q = (torch.randn(T, H, d, device=DEV) * 2 * d ** -0.5).bfloat16()
    meta = AttnMeta(slots=None, block_tables=bt, qstart=qs, qlen=ql, ctx=cx, tile_seq=None, tile_tok0=None, last_idx=None, host_qlen=qlens)
    ts, tt = meta.latent_tiles(1, DEV, seqmix.gqa_tokens_per_tile(H, G, True))
    return q, kc, vc, bt, qs, ql, cx, ts, tt


FORMS = {"plain": {}, "window": {"window": 70}, "kept": {"window": 90, "keep_first": 5}, "chunk": {"chunk": 100}, "cap": {"softcap": 20.0},
         "wide cap": {"softcap": 90.0}, "sink": {"sink": 0.7}, "sinks": {"sinks": 1}, "slopes": {"slopes": 1}}


@pytest.mark.parametrize("H,G,d,dv", [(8, 2, 64, 64), (3, 3, 8, 5), (32, 1, 72, 60), (4, 2, 96, 64), (6, 2, 128, 100), (2, 1, 136, 128), (64, 1, 192, 7)])
@pytest.mark.parametrize("qlens,ctxs", [([130, 17, 33], [130, 81, 400]), ([65], [65]), ([64, 20], [64, 640])])
@pytest.mark.parametrize("form", list(FORMS))
def test_against_64_bits_and_the_other_form(H, G, d, dv, qlens, ctxs, form):
    a = setup(H, G, d, dv, qlens, ctxs)
    q, kc, vc, bt, qs, ql, cx, ts, tt = a
    T, kw = q.shape[0], dict(FORMS[form])
    for k in ("sinks", "slopes"):
        if k in kw:
            kw[k] = torch.rand(H, device=DEV) * (1.0 if k == "sinks" else 0.05)
    wide = torch.randn(T, H * dv + 3, device=DEV).bfloat16()
    for gate, splits in ((None, 1), (wide[:, 1:H * dv + 1], 3), (torch.randn(T, H, device=DEV).bfloat16(), 1)):
        run = lambda **o: seqmix.paged_gqa_attention(*a, gate, mfma=True, splits=splits, **kw, **o)  # noqa: E731
        old = run(out_f32=True)
        got = run()
        odd = torch.zeros(T, H * dv + 5, dtype=torch.bfloat16, device=DEV)
        run(out=odd[:, 2:H * dv + 2])
        assert torch.equal(odd[:, 2:H * dv + 2], got) and not odd[:, :2].any() and not odd[:, H * dv + 2:].any()
        k64 = {k: v.double() if torch.is_tensor(v) else v for k, v in kw.items()}
        want = ref.paged_gqa_attention(q.double(), kc.double(), vc.double(), bt, qs, ql, cx, None if gate is None else gate.double(), k64.get("window", 0),
                                       False, k64.get("keep_first", 0), k64.get("sink", 0.0), k64.get("chunk", 0), k64.get("softcap", 0.0),
                                       k64.get("sinks"), None, k64.get("slopes"))
        err = (old.double() - want).abs()      # weights in two bf16 parts and f32 sums: some 2^-17 of the values' sizes; then one rounding
        size = want.abs().amax(1, keepdim=True).clamp_min(1.0)
        assert (err <= 2.0 ** -14 * size).all()
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * size).all()


def test_no_further_from_64_bits():
    """Rounded to bf16, the form's outputs are no further from the exact ones than the other form's rounded f32 outputs."""
    a = setup(8, 2, 64, 64, [700, 301], [700, 301])
    want = ref.paged_gqa_attention(*(x.double() for x in a[:3]), *a[3:7], None, 0, False, 0, 0.0, 0, 0.0, None, None, None)
    exact = want.to(torch.bfloat16)
    new, old = (seqmix.paged_gqa_attention(*a, None, mfma=True, out_f32=f).to(torch.bfloat16) for f in (False, True))
    miss = [int((x != exact).sum()) for x in (new, old)]
    print("not the bf16 next to the exact value, of %d: %d, other form %d" % (exact.numel(), *miss))
    assert miss[0] <= 1.02 * miss[1] + 20


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_rows_that_see_what_is_not_finite(bad):
    """A value that is not finite is lost to the rows that see its key (and those of its tile of 64 keys, whose weight for it is 0), as in the other
    form, and to no others; a key that is not, to the rows that see it."""
    for cache in (2, 1):
        a = setup(8, 2, 64, 64, [150, 40], [150, 40])
        clean = seqmix.paged_gqa_attention(*a, None, mfma=True)
        if cache == 2:
            a[2][a[3][0, 6].long(), 1, 9, 4] = bad      # sequence 0, key 100, value head 1, dim 9
        else:
            a[1][a[3][0, 6].long(), 1, 4, 9] = bad
        got, old = (seqmix.paged_gqa_attention(*a, None, mfma=True, out_f32=f) for f in (False, True))
        lost = ~got.isfinite().view(190, 2, 4, 64)
        assert torch.equal(lost, ~old.isfinite().view(190, 2, 4, 64))
        assert lost[100:150, 1, :, 9].all() or (cache, bad) == (1, float("inf"))      # (a score of -inf is a weight of 0)
        assert lost.any() and not lost[:, 0].any() and not lost[:64].any() and not lost[150:].any()
        same = ~lost
        if cache == 1:      # (a key of weight 0 instead of its own)
            same[64:150, 1] = False
        assert torch.equal(got.view(190, 2, 4, 64)[same], clean.view(190, 2, 4, 64)[same])


@pytest.mark.parametrize("d,dv", [(64, 64), (96, 64), (128, 128)])
@pytest.mark.parametrize("mean,splits", [(0.0, 1), (20.0, 1), (20.0, 3), (100.0, 1)])
def test_long_contexts_keep_their_oldest_keys_weights(mean, splits, d, dv):
    """Every key of the older half (values 1) is there again in the newer half (values -1), scores `mean` +- 1: outputs near 0 (the newest rows see a few
    keys of the newer half less), and a weight that loses or gains a share a tile is off by all of that share.  Weights are in two bf16 parts: 2^-17 of each at
    most, in any direction; scores are f32 sums, off by some 2^-24 of the largest, alike for a key and its copy."""
    n, T = 24000, 40
    q, kc, vc, bt, qs, ql, cx, ts, tt = setup(4, 2, d, dv, [T], [n])
    q, page = torch.zeros_like(q), bt[0].long()
    q[:, :, 0], q[:, :, 1] = 4.0, 1.0
    half = torch.randn(n // 2, 2, d, device=DEV)
    half[:, :, 0] = mean / 4
    keys = torch.cat([half, half[torch.randperm(n // 2, device=DEV)]]).bfloat16()
    kc[page] = keys.view(-1, 16, 2, d).transpose(1, 2)
    vc[page[:n // 32]], vc[page[n // 32:]] = 1.0, -1.0
    a = (q, kc, vc, bt, qs, ql, cx, ts, tt)
    want = ref.paged_gqa_attention(q.double(), kc.double(), vc.double(), bt, qs, ql, cx, None, 0, False, 0, 0.0, 0, 0.0, None, None, None)
    got, old = (seqmix.paged_gqa_attention(*a, None, mfma=True, splits=splits, out_f32=f) for f in (False, True))
    assert want.abs().max() < 0.02
    err, err_old = ((x.double() - want).abs().max().item() for x in (got, old))
    print("keys %d, scores %g, %d split(s): off by %.2g, other form %.2g" % (n, mean, splits, err, err_old))
    assert err <= 2.0 ** -9 * want.abs().max().item() + 2.0 ** -18


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("splits", [1, 2])
def test_scores_that_leave_f32_times_log2_e(sign, splits):
    """Scores of 2.5e38 and -2.5e38 are f32 numbers and 1.44 times them are not: the row's largest takes all, the rows without one are as ever."""
    q, kc, vc, bt, qs, ql, cx, ts, tt = setup(8, 2, 64, 64, [150, 70], [150, 70])
    q[:, :, 0] = 0.0
    q[64:90, 1, 0] = 2.0 ** 64
    kc[:, :, :, 0] = sign * 2.0 ** 63 * (1.0 + torch.arange(16, device=DEV)[None, None] / 32)      # scores to 2^127 (1 + 15 / 32)
    a = (q, kc.bfloat16(), vc, bt, qs, ql, cx, ts, tt)
    want = ref.paged_gqa_attention(q.double(), kc.double(), vc.double(), bt, qs, ql, cx, None, 0, False, 0, 0.0, 0, 0.0, None, None, None)
    got, old = (seqmix.paged_gqa_attention(*a, None, mfma=True, splits=splits, out_f32=f) for f in (False, True))
    size = want.abs().amax(1, keepdim=True).clamp_min(1.0)
    assert ((old.double() - want).abs() <= 2.0 ** -14 * size).all()
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * size).all()
